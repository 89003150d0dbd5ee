// Split-KV attention of 17 to 32 queries per KV head (a verify pass) over
// page-aligned tiles (page_tokens a multiple of 16) for contexts that fill the
// CUs: both products on int8 MFMA 16x16x64 with exact integer sums. Included
// after paged_attention.hip (page format, the kernels of fewer queries, smaller
// contexts and other page sizes) and qmatvec_tiled.hip (transpose4).
//
// A workgroup takes one KV head and a run of 256-token steps; wave w of a query
// tile loads and scores tokens 64 w .. 64 w + 63 of a step (four 16-token tiles),
// and then owns value dims 64 w .. 64 w + 63 for all of the step's tokens.
//
//  A token's K (V) head run is four blocks, 72 bytes Q2 or 136 Q4: consecutive
//  lanes read its consecutive 8 bytes, and an LDS pass hands lane (li, lg) block
//  lg of token li, scale and codes. (Each lane reading its own block's 16 bytes,
//  18 or 34 apart and 2 off alignment, took about 60 cycles per load: 3.6 us of a
//  256-token step.)
//
//  Scores S = K Q^T, per 64-dim block: a 4 x 4 lane transpose leaves a lane
//  quarter lg of each of its token's blocks, which is its A operand, as bytes
//  2 code. The query is a fixed point X of 22 bits per block, in three balanced
//  int8 limbs, and sum X (2 code - K) (K = 3 Q2, 15 Q4) is formed in
//  int32 exactly: the -K sum X enters as the MFMA's C operand. One conversion
//  and one fma with the block's scale per (token, query, block).
//
//  O^T += V^T P^T: the step's probabilities go through LDS as fp32, and the
//  wave that owns a value block rounds P x (V scale) to a 23-bit fixed point
//  (against the query's largest product of the step) in three int8 limbs: the B
//  operand, whose k order is the one the scores' C layout leaves, so a lane
//  packs its own tokens. The A operand is the codes themselves, dims as rows:
//  ds_read_b64_tr_b4 hands lane l nibble l % 16 of 16 tokens of its choice, a
//  Q4 code or two Q2 codes. Limb sums stay exact in int32 over the whole step;
//  sum X code and sum X (a row of ones) give sum X (2 code - K), one conversion
//  per limb and one fma per step.
//
// The other split, a wave keeping its tokens for both products (as the other
// kernels do), pays the O conversion per wave and merges four O's in LDS; here
// one step's 256 tokens are converted once.
//
// Bound by VALU issue and a long start: 2000 VALU instructions per wave and step
// (the f16 kernel takes 750 per 16-token tile, 3000 for the same tokens), but
// every wave scores four tiles before the first result. 32768 tokens of 24 / 4
// heads, 5 rows: 31.3 us against 39.2 (the combine's 3 us included). (With up to
// 16 queries, 256 threads, it was the faster one only where the steps just fill
// the CUs, by up to 4%; 1 row: 6500 tokens 16.2 us against the f16 kernel's 13.3,
// 16384 16.5 / 16.2, 32768 20.7 / 21.3, 32773 32.5 / 24.3, 131072 59.6 / 53.7.)
// Against float64 the output is off by 1.2e-6 of its norm (the f16 kernel's by
// 1.8e-6; 1.9e-6 and 1 us less with one fixed point per step from the largest V
// scale, which a token of large values and no probability takes from all others).

typedef int pt_v2i __attribute__((ext_vector_type(2)));
#define PT_STEP 256   // tokens per step
#define PT_QT 2       // tiles of 16 queries
#define PT_RS 136     // LDS bytes of one token's V codes (4 blocks of 32, or 16; + 8: the transposed reads of 64
                      // tokens spread over the banks)

struct PtLds {
    int8_t limbs[3][16 * PT_QT][PA_QB];
    uint8_t v[PT_STEP * PT_RS];
    float p[PT_QT][4][4][64][4];         // [query tile][64-token part][token tile][lane][token 4 lg + c]; before
                                     // that a wave's part stages its keys
    float ksc[4 * PT_QT][4][4][16];      // [wave][tile][block][token]: K scale / K
    float vsc[4][PT_STEP];           // [block][token]: V scale
    float smax[4][PT_QT][16];
    uint32_t vmax[4][4];             // [wave][block]: largest |V scale| (bits)
    uint32_t held[4];                // [wave]: whether it has a token
    float4 qs[16 * PT_QT];               // [query], a block each: score per unit of (key scale x integer sum), base 2
    int32_t xs[16 * PT_QT][4];           // [query][block]: sum of X
    float den[4][PT_QT][16];
};

// Bytes of four words, three limbs: l_k holds byte k of z0..z3, as signed digits
// (the words carry + 0x808080).
__device__ __forceinline__ void pt_limbs4(uint32_t z0, uint32_t z1, uint32_t z2, uint32_t z3, uint32_t &l0,
                                          uint32_t &l1, uint32_t &l2) {
    const uint32_t t01 = __builtin_amdgcn_perm(z1, z0, 0x05010400u), t23 = __builtin_amdgcn_perm(z3, z2, 0x05010400u);
    const uint32_t u01 = __builtin_amdgcn_perm(z1, z0, 0x0c0c0602u), u23 = __builtin_amdgcn_perm(z3, z2, 0x06020c0cu);
    l0 = __builtin_amdgcn_perm(t23, t01, 0x05040100u) ^ 0x80808080u;
    l1 = __builtin_amdgcn_perm(t23, t01, 0x07060302u) ^ 0x80808080u;
    l2 = (u01 | u23) ^ 0x80808080u;
}

// Over a row of 16 lanes (DPP rotations, no LDS trip).
__device__ __forceinline__ uint32_t pt_row_umax(uint32_t v) {
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xF, 0xF, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xF, 0xF, false));
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x122, 0xF, 0xF, false));
    return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x121, 0xF, 0xF, false));
}

// Queries to limbs: thread i takes (query, block, quarter) = (i / 16, i / 4 % 4,
// i % 4). X = rint(q 2^E), |X| <= 2^21, E from the query block's largest |q|. A
// quarter's 16 dims are stored as byte 4 j + i of dim 4 i + j, the order in which
// a word's four crumbs (or re-paired nibbles) unpack.
__device__ __forceinline__ void pt_prep(const GqaArgs &a, const float (&q)[16], PtLds &L) {
    const uint32_t i = threadIdx.x, qi = i / 16, b = (i / 4) % 4, part = i % 4;
    float mx = 0.0f;
#pragma unroll
    for (int d = 0; d < 16; d++) mx = fmaxf(mx, fabsf(q[d]));
    mx = fmaxf(mx, __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(mx), 0xB1, 0xF, 0xF, false)));
    mx = fmaxf(mx, __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(mx), 0x4E, 0xF, 0xF, false)));
    int ex = 0;
    frexpf(mx, &ex);  // mx < 2^ex
    const float e = mx > 0.0f ? ldexpf(1.0f, 21 - ex) : 0.0f;
    uint32_t z[16];
    int32_t sum = 0;
#pragma unroll
    for (int d = 0; d < 16; d++) {
        const int32_t X = (int32_t)rintf(q[d] * e);
        sum += X;
        z[d] = (uint32_t)X + 0x808080u;
    }
    uint32_t l[3][4];
#pragma unroll
    for (int j = 0; j < 4; j++) pt_limbs4(z[j], z[4 + j], z[8 + j], z[12 + j], l[0][j], l[1][j], l[2][j]);
#pragma unroll
    for (int k = 0; k < 3; k++)
        *(uint4 *)&L.limbs[k][qi][64 * b + 16 * part] = make_uint4(l[k][0], l[k][1], l[k][2], l[k][3]);
    sum += __builtin_amdgcn_update_dpp(0, sum, 0xB1, 0xF, 0xF, false);  // the quad's lanes
    sum += __builtin_amdgcn_update_dpp(0, sum, 0x4E, 0xF, 0xF, false);
    if (part == 0) {
        L.xs[qi][b] = sum;
        ((float *)&L.qs[qi])[b] = mx > 0.0f ? ldexpf(a.scale * PA_LOG2E, ex - 21) : 0.0f;
    }
}

// Where a wave's four tiles of a step lie (uniform).
struct PtTiles {
    const uint8_t *page[4];
    uint32_t lo[4], hi[4];  // tokens [lo, hi) are held
    uint32_t q4;            // bit i: tile i lies in a Q4 page
};

// desc: lane at + i holds the page of the wave's tile i.
__device__ __forceinline__ void pt_tiles(const GqaArgs &a, const uint4 &desc, uint32_t at, PtTiles &t) {
    t.q4 = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t prec = __builtin_amdgcn_readlane(desc.x, at + i), slot = __builtin_amdgcn_readlane(desc.y, at + i);
        const uint32_t cnt = __builtin_amdgcn_readlane(desc.z, at + i), first = __builtin_amdgcn_readlane(desc.w, at + i);
        t.q4 |= prec != 0 ? 1u << i : 0u;
        t.lo[i] = first;
        t.hi[i] = min(first + cnt, a.tokens);
        t.page[i] = prec != 0 ? a.q4 + (size_t)slot * a.q4_page_bytes : a.q2 + (size_t)slot * a.q2_page_bytes;
    }
}

// 8-byte pieces of a tile's 16 head runs: piece e = 64 n + lane is part e % P of token e / P, P = 9
// (Q2) or 17 (Q4; of a Q2 page's tile there, 9 parts exist). Lanes without a piece or a token read
// the query buffer, which is never used.
template <int N, int P>
__device__ __forceinline__ void pt_load(const GqaArgs &a, const uint8_t *page, uint32_t lo, uint32_t hi, uint32_t tb,
                                        uint32_t run, uint32_t token_bytes, uint32_t parts, uint32_t lane, uint2 (&r)[N]) {
#pragma unroll
    for (int n = 0; n < N; n++) {
        const uint32_t e = 64 * n + lane, tok = e / P, j = tb + tok;
        const bool ok = e < 16 * P && e % P < parts && j >= lo && j < hi;
        const uint8_t *p = ok ? page + (j - lo) * token_bytes + run + 8 * (e % P) : (const uint8_t *)a.query;
        r[n] = make_uint2(((const uint32_t *)p)[0], ((const uint32_t *)p)[1]);
    }
}
// The pieces to rows of PT_RS bytes, and block lg of row li back: its scale and 4 (8) words of codes.
// Block lg starts at bs lg bytes (bs 18 or 34), i.e. its codes at a word or two bytes past one.
template <int N, int P>
__device__ __forceinline__ void pt_stage(uint8_t *rows, uint32_t bs, uint32_t lane, const uint2 (&r)[N],
                                         uint32_t (&codes)[8], uint32_t &scale) {
#pragma unroll
    for (int n = 0; n < N; n++) {
        const uint32_t e = 64 * n + lane;
        if (e < 16 * P) *(uint2 *)(rows + e / P * PT_RS + 8 * (e % P)) = r[n];
    }
    lds_wave_order();
    constexpr int W = P == 9 ? 4 : 8;
    const uint32_t start = (lane >> 4) * bs;
    const uint8_t *row = rows + (lane & 15) * PT_RS;
    scale = *(const uint16_t *)(row + start);
    const uint32_t *w = (const uint32_t *)(row + ((start + 2) & ~3u));
    uint32_t x[W + 1];
#pragma unroll
    for (int i = 0; i <= W; i++) x[i] = w[i];
#pragma unroll
    for (int i = 0; i < W; i++) codes[i] = __builtin_amdgcn_alignbyte(x[i + 1], x[i], (start + 2) & 3u);
    lds_wave_order();  // (the caller writes the rows again)
}

// Q2 codes c as Q4 codes 5 c: (2 * 5 c - 15) / 15 = (2 c - 3) / 3, the same value.
__device__ __forceinline__ uint32_t pt_widen8(uint32_t x) {  // 8 crumbs in the low half
    x = (x | (x << 8)) & 0x00FF00FFu;
    x = (x | (x << 4)) & 0x0F0F0F0Fu;
    x = (x | (x << 2)) & 0x33333333u;
    return x | (x << 2);
}
__device__ __forceinline__ void pt_widen(uint32_t (&c)[8]) {
#pragma unroll
    for (int i = 3; i >= 0; i--) {
        c[2 * i + 1] = pt_widen8(c[i] >> 16);
        c[2 * i] = pt_widen8(c[i] & 0xffffu);
    }
}

// The pages of 64 tiles from `tile` on, one per lane (no tokens past T1 or the page table).
__device__ __forceinline__ uint4 pt_descs(const GqaArgs &a, uint32_t tile, uint32_t T1, uint32_t lane) {
    const uint32_t x = tile + lane, p = x < T1 ? x * 16 / a.page_tokens : a.page_count;
    uint4 d = ((const uint4 *)a.desc)[p < a.page_count ? p : 0];
    if (p >= a.page_count) d.x = d.z = 0;
    return d;
}

// grid (splits, kv heads), 512 threads: waves 4 qt .. 4 qt + 3 serve query tile qt (both quads read the
// keys, the first one's V codes are staged for both). A workgroup takes tiles_per_wave tiles (a multiple of 16) from split * tiles_per_wave on.
// Q4: whether a tile of the workgroup lies in a Q4 page (tiles of Q2 pages are then widened).
template <bool Q4>
__device__ __forceinline__ void pt_run(const GqaArgs &a, PtLds &L, uint32_t T0, uint32_t T1, uint4 desc) {
    const uint32_t lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t li = lane & 15, lg = lane >> 4, h = blockIdx.y, wave = wv & 3, qt = wv >> 2;
    constexpr float inv_k = Q4 ? 1.0f / 15.0f : 1.0f / 3.0f;
    constexpr int32_t neg_k = Q4 ? -15 : -3;
    constexpr uint32_t blk = Q4 ? 32 : 16;  // bytes of a V block's codes
    constexpr int N = Q4 ? 5 : 3;
    const uint32_t qi = 16 * qt + li;
    const int32_t lim = qi < a.queries ? (int32_t)(a.tokens - a.rows + qi / a.group) : -1;
    float m = -INFINITY, den = 0.0f;
    pa_v4f o[4];  // [dim tile]
#pragma unroll
    for (int b = 0; b < 4; b++) o[b] = pa_v4f{0.0f, 0.0f, 0.0f, 0.0f};
    uint8_t *kst = (uint8_t *)&L.p[qt][wave][0][0][0];
    for (uint32_t T = T0; T < T1; T += 16) {
        const uint32_t tb = (T + 4 * wave) * 16, at = (T - T0) & 63;
        if (T != T0 && at == 0) desc = pt_descs(a, T, T1, lane);
        PtTiles t;
        pt_tiles(a, desc, at + 4 * wave, t);
        uint2 kr[4][N], vr[4][N];
        uint32_t piece = lane;
        if (Q4) asm volatile("" : "+v"(piece));  // (its loop invariant offsets would not fit the registers)
        auto load = [&](uint2 (&r)[4][N], uint32_t first) {  // first: of the token's blocks
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const bool q4 = Q4 && ((t.q4 >> i) & 1u);
                pt_load<N, Q4 ? 17 : 9>(a, t.page[i], t.lo[i], t.hi[i], tb + 16 * i, first * (q4 ? 34 : 18),
                                        q4 ? a.q4_token_bytes : a.q2_token_bytes, q4 ? 17 : 9, piece, r[i]);
            }
        };
        load(kr, 4 * h);
        if (qt == 0) load(vr, a.component_values / 64 + 4 * h);
        bool any = false;
        bool whole = tb + 63 + a.rows <= a.tokens;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t b = tb + 16 * i;
            any |= t.hi[i] > t.lo[i] && t.hi[i] > b && t.lo[i] < b + 16;
            whole = whole && t.lo[i] <= b && t.hi[i] >= b + 16;
        }
        // ---- K and V by (token, block); scales and V codes to LDS
        uint32_t kc[4][8];
        auto stage = [&](uint8_t *rows, int i, const uint2 (&r)[N], uint32_t (&c)[8]) {
            uint32_t sc;
            const bool q4 = Q4 && ((t.q4 >> i) & 1u);
            pt_stage<N, Q4 ? 17 : 9>(rows, q4 ? 34 : 18, piece, r, c, sc);
            if (Q4 && !q4) pt_widen(c);
            const uint32_t j = tb + 16 * i + li;
            return pa_half(j >= t.lo[i] && j < t.hi[i] ? sc : 0u);  // absent tokens have a zero scale
        };
#pragma unroll
        for (int i = 0; i < 4; i++) L.ksc[wv][i][lg][li] = stage(kst, i, kr[i], kc[i]) * inv_k;
        if (qt == 0) {
            uint32_t vmx = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint8_t *rows = L.v + (64 * wave + 16 * i) * PT_RS;
                uint32_t c[8];
                const float vs = stage(rows, i, vr[i], c);
                vmx = max(vmx, __float_as_uint(vs) & 0x7fffffffu);  // (a NaN counts as the largest)
                L.vsc[lg][64 * wave + 16 * i + li] = vs;
                uint2 *d = (uint2 *)(rows + li * PT_RS + blk * lg);
#pragma unroll
                for (int x = 0; x < (Q4 ? 4 : 2); x++) d[x] = make_uint2(c[2 * x], c[2 * x + 1]);
            }
            vmx = pt_row_umax(vmx);
            if (li == 0) L.vmax[wave][lg] = vmx;
            if (lane == 0) L.held[wave] = any;
        }
        // ---- scores
        float s[4][4];
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int c = 0; c < 4; c++) s[i][c] = 0.0f;
        if (any) {
            // The query limbs are loop invariant; the opaque offset keeps the
            // compiler from holding all of them in registers across steps.
            uint32_t qoff = qi * PA_QB + 16 * lg;
            asm volatile("" : "+v"(qoff));
            const float4 qs4 = L.qs[qi];
            const float qs[4] = {qs4.x, qs4.y, qs4.z, qs4.w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                if (Q4) {  // quarter q of a block is words 2 q, 2 q + 1
                    transpose4(kc[i][0], kc[i][2], kc[i][4], kc[i][6]);
                    transpose4(kc[i][1], kc[i][3], kc[i][5], kc[i][7]);
                } else {
                    transpose4(kc[i][0], kc[i][1], kc[i][2], kc[i][3]);
                }
            }
#pragma unroll
            for (int b = 0; b < 4; b++) {
                __builtin_amdgcn_sched_barrier(0);  // (a block's results at a time in registers)
                pa_i4 qv[3], ak[4];
                if (Q4) {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const uint32_t x = kc[i][2 * b], y = kc[i][2 * b + 1];
                        const uint32_t xl = (x << 1) & 0x1E1E1E1Eu, xh = (x >> 3) & 0x1E1E1E1Eu;
                        const uint32_t yl = (y << 1) & 0x1E1E1E1Eu, yh = (y >> 3) & 0x1E1E1E1Eu;
                        ak[i] = pa_i4{(int)__builtin_amdgcn_perm(yl, xl, 0x06040200u), (int)__builtin_amdgcn_perm(yh, xh, 0x06040200u),
                                      (int)__builtin_amdgcn_perm(yl, xl, 0x07050301u), (int)__builtin_amdgcn_perm(yh, xh, 0x07050301u)};
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const uint32_t x = kc[i][b];
                        ak[i] = pa_i4{(int)((x << 1) & 0x06060606u), (int)((x >> 1) & 0x06060606u), (int)((x >> 3) & 0x06060606u),
                                      (int)((x >> 5) & 0x06060606u)};
                    }
                }
                const int32_t c0 = neg_k * L.xs[qi][b];
#pragma unroll
                for (int k = 0; k < 3; k++) qv[k] = *(const pa_i4 *)(&L.limbs[k][0][64 * b] + qoff);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float4 f = *(const float4 *)&L.ksc[wv][i][b][4 * lg];
                    const float fb[4] = {f.x * qs[b], f.y * qs[b], f.z * qs[b], f.w * qs[b]};
                    const pa_i4 a0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(ak[i], qv[0], pa_i4{c0, c0, c0, c0}, 0, 0, 0);
                    const pa_i4 a1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(ak[i], qv[1], pa_i4{0, 0, 0, 0}, 0, 0, 0);
                    const pa_i4 a2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(ak[i], qv[2], pa_i4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        const uint32_t u = (uint32_t)a0[c] + ((uint32_t)a1[c] << 8) + ((uint32_t)a2[c] << 16);
                        s[i][c] = fmaf(fb[c], (float)(int32_t)u, s[i][c]);
                    }
                }
            }
        }
        float mt = -INFINITY;
        if (any) {
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int c = 0; c < 4; c++) asm volatile("" : "+v"(s[i][c]));  // (formed here, not in the branch below)
            if (!whole) {
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int c = 0; c < 4; c++) {
                        const uint32_t j = tb + 16 * i + 4 * lg + c;
                        const uint32_t ok = (uint32_t)(j >= t.lo[i]) & (uint32_t)(j < t.hi[i]) & (uint32_t)((int32_t)j <= lim);
                        s[i][c] = ok ? s[i][c] : -INFINITY;
                    }
            }
#pragma unroll
            for (int i = 0; i < 4; i++) mt = fmaxf(mt, fmaxf(fmaxf(s[i][0], s[i][1]), fmaxf(s[i][2], s[i][3])));
        }
        mt = pa_max_x32(pa_max_x16(mt));
        if (lg == 0) L.smax[wave][qt][li] = mt;
        lds_barrier();
        float mn = m;
#pragma unroll
        for (int w = 0; w < 4; w++) mn = fmaxf(mn, L.smax[w][qt][li]);
        const float ref = mn == -INFINITY ? 0.0f : mn;  // (nothing visible yet)
        const float alpha = __builtin_amdgcn_exp2f(m - ref);
        m = mn;
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float4 p = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (any)
                p = make_float4(__builtin_amdgcn_exp2f(s[i][0] - ref), __builtin_amdgcn_exp2f(s[i][1] - ref),
                                __builtin_amdgcn_exp2f(s[i][2] - ref), __builtin_amdgcn_exp2f(s[i][3] - ref));
            sum += (p.x + p.y) + (p.z + p.w);
            *(float4 *)&L.p[qt][wave][i][lane][0] = p;
        }
        den = den * alpha + sum;
        const uint32_t vb = max(max(L.vmax[0][wave], L.vmax[1][wave]), max(L.vmax[2][wave], L.vmax[3][wave]));
        lds_barrier();
        // P x (scale of value block `wave`) of the lane's tokens, and the query's fixed point: 2^e above the
        // largest product, so that a token of large values and little probability takes no bits from the others.
        float pv[4][16], mx = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; w++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float4 p = *(const float4 *)&L.p[qt][w][i][lane][0];
                const float4 v = *(const float4 *)&L.vsc[wave][64 * w + 16 * i + 4 * lg];
                const float pp[4] = {p.x, p.y, p.z, p.w}, vv[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int c = 0; c < 4; c++) pv[w][4 * i + c] = pp[c] * vv[c];
#pragma unroll
                for (int c = 0; c < 4; c += 2)
                    mx = fmaxf(fmaxf(mx, fabsf(pv[w][4 * i + c])), fabsf(pv[w][4 * i + c + 1]));
            }
        mx = pa_max_x32(pa_max_x16(mx));
        const int ex = min(max((int)(__float_as_uint(mx) >> 23) - 126, -100), 17);
        const float to_x = __uint_as_float((uint32_t)(127 + 22 - ex) << 23);
        const float back = vb < 0x7f800000u ? __uint_as_float((uint32_t)(127 - 22 + ex) << 23) : __builtin_nanf("");
        // ---- O^T of the block over the step's tokens
        const uint32_t vrow = (16 * (li >> 2) + 4 * lg + (li & 3)) * PT_RS + blk * wave;
        pa_i4 acc[4][3], ones[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            ones[k] = pa_i4{0, 0, 0, 0};
#pragma unroll
            for (int d = 0; d < 4; d++) acc[d][k] = pa_i4{0, 0, 0, 0};
        }
#pragma unroll
        for (int w = 0; w < 4; w++) {
            if (!__builtin_amdgcn_readfirstlane(L.held[w])) continue;
            // The sum's low mantissa bits are X + 2^22; + 0x408080 makes it X + 0x808080 (low 24 bits).
            uint32_t z[16];
#pragma unroll
            for (int x = 0; x < 16; x++) z[x] = __float_as_uint(fmaf(pv[w][x], to_x, 12582912.0f)) + 0x408080u;
            uint32_t l[3][4];
#pragma unroll
            for (int x = 0; x < 4; x++) {  // tokens in the order the nibbles unpack: even, odd, of 8 each
                const int i0 = 8 * (x >> 1) + (x & 1);
                pt_limbs4(z[i0], z[i0 + 2], z[i0 + 4], z[i0 + 6], l[0][x], l[1][x], l[2][x]);
            }
            pa_i4 bl[3];
#pragma unroll
            for (int k = 0; k < 3; k++) {
                bl[k] = pa_i4{(int)l[k][0], (int)l[k][1], (int)l[k][2], (int)l[k][3]};
                ones[k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(pa_i4{0x01010101, 0x01010101, 0x01010101, 0x01010101}, bl[k],
                                                                ones[k], 0, 0, 0);
            }
            const uint8_t *vbase = L.v + 64 * w * PT_RS + vrow;
            auto read = [&](int j) {
                return __builtin_amdgcn_ds_read_tr4_b64_v2i32((__attribute__((address_space(3))) pt_v2i *)(vbase + 8 * j));
            };
            pa_i4 av[4];
            if (Q4) {
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    const pt_v2i x = read(d);
                    av[d] = pa_i4{x[0] & 0x0F0F0F0F, (int)((uint32_t)x[0] >> 4) & 0x0F0F0F0F, x[1] & 0x0F0F0F0F,
                                  (int)((uint32_t)x[1] >> 4) & 0x0F0F0F0F};
                }
            } else {
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const pt_v2i x = read(j);
                    const uint32_t x0 = (uint32_t)x[0], x1 = (uint32_t)x[1];
                    av[2 * j] = pa_i4{(int)(x0 & 0x03030303u), (int)((x0 >> 4) & 0x03030303u), (int)(x1 & 0x03030303u),
                                      (int)((x1 >> 4) & 0x03030303u)};
                    av[2 * j + 1] = pa_i4{(int)((x0 >> 2) & 0x03030303u), (int)((x0 >> 6) & 0x03030303u),
                                          (int)((x1 >> 2) & 0x03030303u), (int)((x1 >> 6) & 0x03030303u)};
                }
            }
#pragma unroll
            for (int d = 0; d < 4; d++)
#pragma unroll
                for (int k = 0; k < 3; k++)
                    acc[d][k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[d], bl[k], acc[d][k], 0, 0, 0);
        }
        const float f = back * inv_k;
        const int32_t n01 = neg_k * (ones[0][0] + (ones[1][0] << 8)), n2 = neg_k * ones[2][0];
#pragma unroll
        for (int d = 0; d < 4; d++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                // The low two limbs' sums are below 2^20: joined in int32.
                const float t01 = (float)(2 * (acc[d][0][c] + (acc[d][1][c] << 8)) + n01);
                const float t2 = (float)(2 * acc[d][2][c] + n2);
                o[d][c] = fmaf(fmaf(t2, 65536.0f, t01), f, o[d][c] * alpha);
            }
        lds_barrier();  // the step's LDS is free
    }
    // ---- partial rows and their (maximum, denominator)
    den += __shfl_xor(den, 16);
    den += __shfl_xor(den, 32);
    if (lg == 0) L.den[wave][qt][li] = den;
    lds_barrier();
    const size_t base = ((size_t)h * a.splits + blockIdx.x) * a.queries;
    const float dn = (L.den[0][qt][li] + L.den[1][qt][li]) + (L.den[2][qt][li] + L.den[3][qt][li]);
    const float bad = dn - dn;  // NaN where a score was not finite: the integer sums carry no NaN
    if (qi >= a.queries) return;
    float *dst = a.part_out + (base + qi) * PA_HD + 64 * wave;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (Q4) {  // tile j, row 4 lg + c is dim 16 j + 4 lg + c
            *(float4 *)(dst + 16 * j + 4 * lg) = make_float4(o[j][0] + bad, o[j][1] + bad, o[j][2] + bad, o[j][3] + bad);
        } else {   // tile 2 x + par, row 4 lg + c is dim 32 x + 2 (4 lg + c) + par
            const int x = j >> 1, y = 2 * (j & 1);
            *(float4 *)(dst + 32 * x + 8 * lg + 2 * y) = make_float4(o[2 * x][y] + bad, o[2 * x + 1][y] + bad,
                                                                     o[2 * x][y + 1] + bad, o[2 * x + 1][y + 1] + bad);
        }
    }
    if (wave == 0 && lg == 0) {
        a.part_stats[2 * (base + qi)] = m * PA_LN2;  // the combine works in natural units
        a.part_stats[2 * (base + qi) + 1] = dn;
    }
}

extern "C" __global__ __launch_bounds__(256 * PT_QT, 1) void ctox_paged_gqa_tiles_gfx950(GqaArgs a) {
    __shared__ __align__(16) PtLds L;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t T0 = blockIdx.x * a.tiles_per_wave, T1 = min(T0 + a.tiles_per_wave, a.tiles);
    const uint4 desc = pt_descs(a, T0, T1, lane);
    float qv[1][16];
    pa_prep_load<1>(a, blockIdx.y, qv);
    bool q4 = desc.x != 0;
    for (uint32_t T = T0 + 64; T < T1; T += 64) q4 = q4 || pt_descs(a, T, T1, lane).x != 0;
    pt_prep(a, qv[0], L);
    lds_barrier();
    if (__builtin_amdgcn_ballot_w64(q4) == 0) pt_run<false>(a, L, T0, T1, desc);
    else pt_run<true>(a, L, T0, T1, desc);
}
