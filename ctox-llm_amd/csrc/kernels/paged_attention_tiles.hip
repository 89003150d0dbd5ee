// Split-KV attention over page-aligned tiles (page_tokens a multiple of 16):
// both products on int8 MFMA 16x16x64 with exact integer sums. Included after
// paged_attention.hip (page format and the other page sizes' kernel) and
// qmatvec_tiled.hip (transpose4).
//
// A workgroup takes one KV head and a run of 256-token steps; wave w loads and
// scores tokens 64 w .. 64 w + 63 of a step (four 16-token tiles), and then
// owns value dims 64 w .. 64 w + 63 for all of the step's tokens.
//
//  Scores S = K Q^T, per 64-dim block: lane (li, lg) reads token li's block lg
//  whole (16 B of Q2 codes or 32 B of Q4, straight from the page); a 4 x 4 lane
//  transpose leaves it quarter lg of every block, which is its A operand, as
//  bytes 2 code. The query is a fixed point X of 22 bits per query row, in three
//  balanced int8 limbs, and sum X (2 code - K) (K = 3 Q2, 15 Q4) is formed in
//  int32 exactly: the -K sum X enters as the MFMA's C operand. One conversion
//  and one fma with the block's scale per (token, query, block).
//
//  O^T += V^T P^T: the step's probabilities go through LDS as fp32, and the
//  wave that owns a value block rounds P x (V scale) to a 23-bit fixed point
//  (against the block's largest scale in the step) in three int8 limbs: the B
//  operand, whose k order is the one the scores' C layout leaves, so a lane
//  packs its own tokens. The A operand is the codes themselves, dims as rows:
//  ds_read_b64_tr_b4 hands lane l nibble l % 16 of 16 tokens of its choice, a
//  Q4 code or two Q2 codes. Limb sums stay exact in int32 over the whole step;
//  sum X code and sum X (a row of ones) give sum X (2 code - K), one conversion
//  per limb and one fma per step.
//
// The other split, a wave keeping its tokens for both products (as the fp32
// kernel does), pays the O conversion per wave and merges four O's in LDS; here
// one step's 256 tokens are converted once.
//
// Bound by VALU issue: about 1200 instructions per wave and 256-token step (the
// f16-MFMA kernel before took 750 per 16-token tile, 3000 for the same tokens).

typedef int pt_v2i __attribute__((ext_vector_type(2)));
struct __attribute__((packed, aligned(2))) PtCodes {  // 16 bytes of codes: they follow a 2-byte scale
    uint32_t x[4];
};

#define PT_STEP 256   // tokens per step
#define PT_RS2 72     // LDS bytes of one token's V codes (4 blocks): Q2 (64 + 8: the transposed reads of
#define PT_RS4 136    // 64 tokens spread over the banks), Q4

template <int R>
struct PtLds {
    int8_t limbs[3][16 * R][PA_QB];
    uint8_t v[PT_STEP * PT_RS4];
    float p[R][4][4][64][4];         // [query tile][64-token part][token tile][lane][token 4 lg + c]
    float ksc[4 * R][4][4][16];      // [wave][tile][block][token]: K scale / K
    float vsc[4][PT_STEP];           // [block][token]: V scale
    float smax[4][R][16];
    uint32_t vmax[4][4];             // [wave][block]: largest |V scale| (bits)
    uint32_t held[4];                // [wave]: whether it has a token
    float qs[16 * R];                // score per unit of (block scale x integer sum), base 2
    int32_t xs[16 * R][4];           // [query][block]: sum of X
    float den[4][R][16];
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

// Queries to limbs: thread i takes (query, block, quarter) = (i / 16, i / 4 % 4,
// i % 4). X = rint(q 2^E), |X| <= 2^21, E from the query row's largest |q|. A
// quarter's 16 dims are stored as byte 4 j + i of dim 4 i + j, the order in which
// a word's four crumbs (or re-paired nibbles) unpack.
template <int R>
__device__ __forceinline__ void pt_prep(const GqaArgs &a, const float (&q)[16], PtLds<R> &L) {
    const uint32_t i = threadIdx.x, qi = i / 16, b = (i / 4) % 4, part = i % 4;
    float mx = 0.0f;
#pragma unroll
    for (int d = 0; d < 16; d++) mx = fmaxf(mx, fabsf(q[d]));
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
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
    sum += __shfl_xor(sum, 1);
    sum += __shfl_xor(sum, 2);
    if (part == 0) L.xs[qi][b] = sum;
    if (b == 0 && part == 0) L.qs[qi] = mx > 0.0f ? ldexpf(a.scale * PA_LOG2E, ex - 21) : 0.0f;
}

// One wave's four tiles of a step in registers.
struct PtTiles {
    PtCodes k[4][2], v[4][2];   // [tile][second half: Q4 only]
    uint16_t ks[4], vs[4];      // fp16 scales of (token li, block lg)
    uint32_t lo[4], hi[4];      // tokens [lo, hi) of the tile's page are held (uniform)
    uint32_t q4;                // tiles in Q4 pages (uniform bits)
};

// Q2 codes c as Q4 codes 5 c: (2 * 5 c - 15) / 15 = (2 c - 3) / 3, the same value.
__device__ __forceinline__ uint32_t pt_widen8(uint32_t x) {  // 8 crumbs in the low half
    x = (x | (x << 8)) & 0x00FF00FFu;
    x = (x | (x << 4)) & 0x0F0F0F0Fu;
    x = (x | (x << 2)) & 0x33333333u;
    return x | (x << 2);
}
__device__ __forceinline__ void pt_widen(PtCodes (&c)[2]) {
    uint32_t w[8];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        w[2 * i] = pt_widen8(c[0].x[i] & 0xffffu);
        w[2 * i + 1] = pt_widen8(c[0].x[i] >> 16);
    }
#pragma unroll
    for (int i = 0; i < 8; i++) c[i / 4].x[i % 4] = w[i];
}

// Q4: 0 no tile of the workgroup lies in a Q4 page; 1 some do, and tiles of Q2 pages are widened.
// desc: lane i < 4 holds the page of the wave's tile i. A lane without a token reads the query
// buffer, which is never used.
template <int Q4>
__device__ __forceinline__ void pt_load(const GqaArgs &a, const uint4 &desc, uint32_t tb, uint32_t h, uint32_t li,
                                        uint32_t lg, PtTiles &t) {
    t.q4 = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t prec = __builtin_amdgcn_readlane(desc.x, i), slot = __builtin_amdgcn_readlane(desc.y, i);
        const uint32_t cnt = __builtin_amdgcn_readlane(desc.z, i), first = __builtin_amdgcn_readlane(desc.w, i);
        const bool q4 = Q4 && prec != 0;
        t.q4 |= q4 ? 1u << i : 0u;
        t.lo[i] = first;
        t.hi[i] = min(first + cnt, a.tokens);
        const uint32_t bs = q4 ? 34u : 18u, j = tb + 16 * i + li;
        const uint8_t *page = q4 ? a.q4 + (size_t)slot * a.q4_page_bytes : a.q2 + (size_t)slot * a.q2_page_bytes;
        const bool ok = j >= t.lo[i] && j < t.hi[i];
        const uint8_t *kp = ok ? page + (j - first) * (q4 ? a.q4_token_bytes : a.q2_token_bytes) + (4 * h + lg) * bs
                               : (const uint8_t *)a.query;
        const uint8_t *vp = ok ? kp + (a.component_values / 64) * bs : kp;
        t.ks[i] = *(const uint16_t *)kp;
        t.vs[i] = *(const uint16_t *)vp;
        t.k[i][0] = *(const PtCodes *)(kp + 2);
        t.v[i][0] = *(const PtCodes *)(vp + 2);
        if (Q4) {
            t.k[i][1] = *(const PtCodes *)(kp + (q4 ? 18 : 2));
            t.v[i][1] = *(const PtCodes *)(vp + (q4 ? 18 : 2));
        }
        if (!ok) t.ks[i] = t.vs[i] = 0;
    }
}

// grid (splits, kv heads), 256 R threads, R = 1 or 2 tiles of 16 queries: waves 4 qt .. 4 qt + 3 serve
// query tile qt (both quads read the keys, the first one's V codes are staged for both). A workgroup
// takes tiles_per_wave tiles (a multiple of 16) from split * tiles_per_wave on.
template <int R, int Q4>
__device__ __forceinline__ void pt_run(const GqaArgs &a, PtLds<R> &L, uint32_t T0, uint32_t T1, uint4 dnext, PtTiles &t) {
    constexpr uint32_t RS = Q4 ? PT_RS4 : PT_RS2;
    const uint32_t lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t li = lane & 15, lg = lane >> 4, h = blockIdx.y, wave = wv & 3, qt = wv >> 2;
    auto desc_of = [&](uint32_t tile) {  // lane i < 4: page of tile + i (no tokens past T1 or the page table)
        const uint32_t x = tile + (lane & 3), p = x < T1 ? x * 16 / a.page_tokens : a.page_count;
        const uint4 d = ((const uint4 *)a.desc)[p < a.page_count ? p : 0];
        return p < a.page_count ? d : make_uint4(0, 0, 0, 0);
    };
    const uint32_t qi = 16 * qt + li;
    const int32_t lim = qi < a.queries ? (int32_t)(a.tokens - a.rows + qi / a.group) : -1;
    const float qs = L.qs[qi];
    float m = -INFINITY, den = 0.0f;
    int32_t xs[4];
    pa_v4f o[4];  // [dim tile]
#pragma unroll
    for (int b = 0; b < 4; b++) {
        xs[b] = L.xs[qi][b];
        o[b] = pa_v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
    for (uint32_t T = T0; T < T1; T += 16) {
        const uint32_t tb = (T + 4 * wave) * 16;
        bool any = false;
        bool whole = tb + 63 + a.rows <= a.tokens;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t b = tb + 16 * i;
            any |= t.hi[i] > t.lo[i] && t.hi[i] > b && t.lo[i] < b + 16;
            whole = whole && t.lo[i] <= b && t.hi[i] >= b + 16;
            if (Q4 && !((t.q4 >> i) & 1u)) {
                pt_widen(t.k[i]);
                pt_widen(t.v[i]);
            }
        }
        // ---- scales and V codes to LDS
        uint32_t vmx = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float vs = pa_half(t.vs[i]);
            vmx = max(vmx, __float_as_uint(vs) & 0x7fffffffu);  // (a NaN counts as the largest)
            L.ksc[wv][i][lg][li] = pa_half(t.ks[i]) * (Q4 ? 1.0f / 15.0f : 1.0f / 3.0f);
            if (qt) continue;
            L.vsc[lg][64 * wave + 16 * i + li] = vs;
            uint2 *d = (uint2 *)(L.v + (64 * wave + 16 * i + li) * RS + (Q4 ? 32 : 16) * lg);
#pragma unroll
            for (int x = 0; x < (Q4 ? 2 : 1); x++) {
                d[2 * x] = make_uint2(t.v[i][x].x[0], t.v[i][x].x[1]);
                d[2 * x + 1] = make_uint2(t.v[i][x].x[2], t.v[i][x].x[3]);
            }
        }
#pragma unroll
        for (int x = 1; x < 16; x <<= 1) vmx = max(vmx, (uint32_t)__shfl_xor((int)vmx, x));
        if (qt == 0 && li == 0) L.vmax[wave][lg] = vmx;
        if (qt == 0 && lane == 0) L.held[wave] = any;
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
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint32_t *k0 = t.k[i][0].x, *k1 = t.k[i][1].x;
                if (Q4) {  // quarter q of a block is words 2 q, 2 q + 1
                    uint32_t e0 = k0[0], e1 = k0[2], e2 = k1[0], e3 = k1[2], f0 = k0[1], f1 = k0[3], f2 = k1[1], f3 = k1[3];
                    transpose4(e0, e1, e2, e3);
                    transpose4(f0, f1, f2, f3);
                    k0[0] = e0; k0[1] = e1; k0[2] = e2; k0[3] = e3;
                    k1[0] = f0; k1[1] = f1; k1[2] = f2; k1[3] = f3;
                } else {
                    transpose4(k0[0], k0[1], k0[2], k0[3]);
                }
            }
#pragma unroll
            for (int b = 0; b < 4; b++) {
                __builtin_amdgcn_sched_barrier(0);  // (a block's results at a time in registers)
                pa_i4 qv[3];
#pragma unroll
                for (int k = 0; k < 3; k++) qv[k] = *(const pa_i4 *)(&L.limbs[k][0][64 * b] + qoff);
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    pa_i4 ak;
                    if (Q4) {
                        const uint32_t x = t.k[i][0].x[b], y = t.k[i][1].x[b];
                        const uint32_t xl = (x << 1) & 0x1E1E1E1Eu, xh = (x >> 3) & 0x1E1E1E1Eu;
                        const uint32_t yl = (y << 1) & 0x1E1E1E1Eu, yh = (y >> 3) & 0x1E1E1E1Eu;
                        ak = pa_i4{(int)__builtin_amdgcn_perm(yl, xl, 0x06040200u), (int)__builtin_amdgcn_perm(yh, xh, 0x06040200u),
                                   (int)__builtin_amdgcn_perm(yl, xl, 0x07050301u), (int)__builtin_amdgcn_perm(yh, xh, 0x07050301u)};
                    } else {
                        const uint32_t x = t.k[i][0].x[b];
                        ak = pa_i4{(int)((x << 1) & 0x06060606u), (int)((x >> 1) & 0x06060606u), (int)((x >> 3) & 0x06060606u),
                                   (int)((x >> 5) & 0x06060606u)};
                    }
                    const float4 f = *(const float4 *)&L.ksc[wv][i][b][4 * lg];
                    const float fb[4] = {f.x, f.y, f.z, f.w};
                    const int32_t c0 = (Q4 ? -15 : -3) * xs[b];
                    const pa_i4 a0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(ak, qv[0], pa_i4{c0, c0, c0, c0}, 0, 0, 0);
                    const pa_i4 a1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(ak, qv[1], pa_i4{0, 0, 0, 0}, 0, 0, 0);
                    const pa_i4 a2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(ak, qv[2], pa_i4{0, 0, 0, 0}, 0, 0, 0);
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
                for (int c = 0; c < 4; c++) {
                    s[i][c] *= qs;
                    asm volatile("" : "+v"(s[i][c]));  // (formed here, not in the branch below)
                }
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
        // The next step's loads go out while this one's probabilities are
        // exchanged (Q4's, twice the registers, after the value product).
        const bool more = T + 16 < T1;
        auto next = [&] {
            pt_load<Q4>(a, dnext, (T + 16 + 4 * wave) * 16, h, li, lg, t);
            dnext = desc_of(T + 32 + 4 * wave);
        };
        if (!Q4 && more) next();
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
        lds_barrier();
        // ---- O^T of value block `wave` over the step's tokens
        uint32_t vb = max(max(L.vmax[0][wave], L.vmax[1][wave]), max(L.vmax[2][wave], L.vmax[3][wave]));
        vb = __builtin_amdgcn_readfirstlane(vb);
        const int ex = min(max((int)(vb >> 23) - 126, -24), 17);  // fp16 scales below 2^ex
        const float sc = ldexpf(1.0f, 22 - ex);
        const float back = vb < 0x7f800000u ? ldexpf(1.0f, ex - 22) : __builtin_nanf("");
        const uint32_t vrow = (16 * (li >> 2) + 4 * lg + (li & 3)) * RS;
        pa_i4 acc[4][3], ones[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            ones[k] = pa_i4{0, 0, 0, 0};
#pragma unroll
            for (int d = 0; d < 4; d++) acc[d][k] = pa_i4{0, 0, 0, 0};
        }
        for (int w = 0; w < 4; w++) {
            if (!__builtin_amdgcn_readfirstlane(L.held[w])) continue;
            uint32_t z[16];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float4 p = *(const float4 *)&L.p[qt][w][i][lane][0];
                const float4 v = *(const float4 *)&L.vsc[wave][64 * w + 16 * i + 4 * lg];
                const float pp[4] = {p.x, p.y, p.z, p.w}, vv[4] = {v.x, v.y, v.z, v.w};
                // The sum's low mantissa bits are X + 2^22; + 0x408080 makes it X + 0x808080 (low 24 bits).
#pragma unroll
                for (int c = 0; c < 4; c++) z[4 * i + c] = __float_as_uint(fmaf(pp[c], vv[c] * sc, 12582912.0f)) + 0x408080u;
            }
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
            const uint8_t *vbase = L.v + 64 * w * RS + vrow + (Q4 ? 32 : 16) * wave;
#pragma unroll
            for (int j = 0; j < (Q4 ? 4 : 2); j++) {
                const pt_v2i x = __builtin_amdgcn_ds_read_tr4_b64_v2i32(
                    (__attribute__((address_space(3))) pt_v2i *)(vbase + 8 * j));
                const uint32_t x0 = (uint32_t)x[0], x1 = (uint32_t)x[1];
#pragma unroll
                for (int par = 0; par < (Q4 ? 1 : 2); par++) {
                    const uint32_t mask = Q4 ? 0x0F0F0F0Fu : 0x03030303u;
                    const pa_i4 av = {(int)((x0 >> (2 * par)) & mask), (int)((x0 >> (4 + 2 * par)) & mask),
                                      (int)((x1 >> (2 * par)) & mask), (int)((x1 >> (4 + 2 * par)) & mask)};
                    const int d = Q4 ? j : 2 * j + par;
#pragma unroll
                    for (int k = 0; k < 3; k++)
                        acc[d][k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bl[k], acc[d][k], 0, 0, 0);
                }
            }
        }
        if (Q4 && more) next();
        const float f = back * (Q4 ? 1.0f / 15.0f : 1.0f / 3.0f);
        int32_t n[3];
#pragma unroll
        for (int k = 0; k < 3; k++) n[k] = (Q4 ? -15 : -3) * ones[k][0];
#pragma unroll
        for (int d = 0; d < 4; d++)
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const float t0 = (float)(2 * acc[d][0][c] + n[0]), t1 = (float)(2 * acc[d][1][c] + n[1]);
                const float t2 = (float)(2 * acc[d][2][c] + n[2]);
                o[d][c] = fmaf(fmaf(t2, 65536.0f, fmaf(t1, 256.0f, t0)), f, o[d][c] * alpha);
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

template <int R>
__device__ __forceinline__ void paged_gqa_tiles(const GqaArgs &a) {
    __shared__ __align__(16) PtLds<R> L;
    const uint32_t lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 3;
    const uint32_t li = lane & 15, lg = lane >> 4, h = blockIdx.y;
    const uint32_t T0 = blockIdx.x * a.tiles_per_wave, T1 = min(T0 + a.tiles_per_wave, a.tiles);
    // Any Q4 page in the workgroup's range? (lanes stride over its tiles)
    bool q4 = false;
    for (uint32_t x = T0 + lane; x < T1; x += 64) {
        const uint32_t p = x * 16 / a.page_tokens;
        q4 = q4 || (p < a.page_count && a.desc[p].precision != 0);
    }
    auto desc_of = [&](uint32_t tile) {
        const uint32_t x = tile + (lane & 3), p = x < T1 ? x * 16 / a.page_tokens : a.page_count;
        const uint4 d = ((const uint4 *)a.desc)[p < a.page_count ? p : 0];
        return p < a.page_count ? d : make_uint4(0, 0, 0, 0);
    };
    const uint4 d0 = desc_of(T0 + 4 * wave), d1 = desc_of(T0 + 16 + 4 * wave);
    float qv[1][16];
    pa_prep_load<1>(a, h, qv);
    PtTiles t;
    // The first step's loads are in flight while the queries are split.
    if (__builtin_amdgcn_ballot_w64(q4) == 0) {
        pt_load<0>(a, d0, (T0 + 4 * wave) * 16, h, li, lg, t);
        pt_prep<R>(a, qv[0], L);
        lds_barrier();
        pt_run<R, 0>(a, L, T0, T1, d1, t);
    } else {
        pt_load<1>(a, d0, (T0 + 4 * wave) * 16, h, li, lg, t);
        pt_prep<R>(a, qv[0], L);
        lds_barrier();
        pt_run<R, 1>(a, L, T0, T1, d1, t);
    }
}

extern "C" __global__ __launch_bounds__(256, 2) void ctox_paged_gqa_tiles_r1_gfx950(GqaArgs a) { paged_gqa_tiles<1>(a); }
extern "C" __global__ __launch_bounds__(512, 1) void ctox_paged_gqa_tiles_r2_gfx950(GqaArgs a) { paged_gqa_tiles<2>(a); }
