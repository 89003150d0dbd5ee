// Chunked (WY-form) gated-delta prefill, gfx950.
//
// The token recurrence of Q/src/reference.rs:230-297 / 377-415,
//   S_t = a_t (I - b_t k_t k_t^T) S_{t-1} + b_t k_t v_t^T,   o_t = S_t^T q_t
// (k, q L2-normalised, q also scaled by 1/sqrt(key_dim), a_t = exp(log_decay_t),
// b_t = beta_t), is evaluated chunk by chunk. Within a chunk of C tokens, with
// G_t = sum_{s<=t} log_decay_s (relative to the chunk start) and g_t = exp(G_t):
//   S_t = g_t S_0 + sum_{r<=t} exp(G_t - G_r) k_r d_r^T
//   d_s = b_s (v_s - g_s S_0^T k_s - sum_{r<s} exp(G_s - G_r) (k_s.k_r) d_r).
// With L the strictly lower b_s exp(G_s - G_r) (k_s.k_r) and T = (I + L)^{-1},
// this is
//   D   = U - W S_0,   U = T diag(b) V,   W = T diag(b g) K
//   O   = diag(g) Q S_0 + A D,       A[t][r] = exp(G_t - G_r) (q_t.k_r), r <= t
//   S_C = g_C S_0 + sum_r exp(G_C - G_r) k_r d_r^T.
// Every decay factor is exp of a non-positive difference for decays <= 1, so
// nothing overflows however strong the decay. (The decay belongs in the
// inverse: that of the undecayed I + L grows as (beta - 1)^n for beta > 2.)
// Only D and S_C depend on the chunks before, so all of W, U, A and the scaled
// rows of Q and K are made for every chunk in parallel (pass 1) and the sequential pass 2 is two small
// products deep per chunk.
//
// Pass 1 (ctox_gdn_chunk_prep_gfx950, one workgroup per (head, chunk)): fp32
// MFMA throughout; T by blocks: the four 16 x 16 diagonal blocks by forward
// substitution (a wave each), the blocks below them on MFMA one block row at a
// time. Its matrices leave as MFMA operands, see below.
// Pass 2 (ctox_gdn_chunk_scan{1,2}_gfx950, one workgroup per (head, 16 or 32
// value columns), chunks in order). Value columns are independent, so slices
// need no exchange. Padded tokens of a partial chunk have k = q = v = 0,
// beta = 0 and log_decay = 0: identity steps.
//
// Pass 2's products run on v_mfma_f32_16x16x32_bf16 with every operand as the
// exact sum of three bf16 parts (24 significant bits, fp32's exponents: no
// scales, whatever the magnitudes of neighbouring tokens, keys or columns are)
// and the six products of parts above 2^-24, accumulated in fp32: 2.7 times the
// fp32 MFMA rate. (Two f16 parts under powers of two per row and column take
// half the MFMAs, but elements 2^17 below their row's or column's largest lose
// bits that fp32 keeps.)
//
// Pass 2 is a latency chain: per chunk the state operand, W S_0, D, its
// exchange, K^T D. Four waves hold the state (fp32, in registers: wave w rows
// 32 w .. 32 w + 31) and walk that chain; four more compute the outputs beside
// them from the same two exchanges. The contraction index order of an operand
// is free as long as both sides agree, and it is chosen so that a lane's MFMA
// results are the very elements of its next operand: no transposes. Nothing
// but the 12 KB state and 6 KB D operands passes through LDS; pass 1's operands
// are read from memory in fragment order, one chunk ahead, straight to
// registers, a few at a time between the chunk's products: 172 KB per chunk and
// CU take 1.1 us of the CU's load path at 64 bytes per clock, which issued in one
// go would come on top of the products' time.
// 4096 tokens of 32 heads: 284 us (under the tracer three launches of 47 us each
// for pass 1 and for pass 2), against 359 for the same chunk algorithm with all of T (b V - b g K
// S_0), Q S_0 + A D and the state update as fp32 MFMA in the sequential pass, and
// 223 with two f16 parts per operand. Error against float64, relative norm:
// outputs 8.4e-7 (fp32 MFMA 8.4e-7), state 1.5e-6 (1.5e-6); 200 tokens of 48
// heads, state 1.6e-7 (fp32 1.7e-7, two f16 parts 1.8e-7). One and
// two chunks gain little from pass 1's extra work: 64 tokens 23.7 us, 128 tokens
// 26.4, with fp32 22.9 and 27.9.

#include <hip/hip_runtime.h>

#include "kernel_args.h"
#include "lds_barrier.h"

#define GC 64        // max chunk length
#define TPAD 65      // LDS row stride of L / T
#define SPAD 132     // LDS row stride of K / Q rows

typedef float gv4f __attribute__((ext_vector_type(4)));
typedef __bf16 gb2 __attribute__((ext_vector_type(2)));
typedef __bf16 gb8 __attribute__((ext_vector_type(8)));

// Scratch of one (head, chunk), byte offsets. A fragment is one MFMA operand
// of 16 rows x 32 contraction elements, [part 3][lane][8 bf16]: lane (m = lane %
// 16, g = lane / 16) holds row m's elements 4 g .. 4 g + 3 and 16 + 4 g .. + 3 of
// the 32 (the order in which two 16 x 16 results hold them).
#define GF_W 0                  // [token strip 4][key step 4] fragments of 3 KB
#define GF_K 49152              // K^T: [key tile 8][token step 2]
#define GF_Q 98304              // as GF_W
#define GF_A 147456             // [token strip 4][token step 2]
#define GF_U 172032             // fp32 [value tile 8][token strip 4][64 lanes][4 rows]
#define GF_AUX 204800           // floats: fq[64], gC
static_assert(GF_AUX + 65 * 4 <= CTOX_GDN_CHUNK_BYTES, "chunk scratch");

__device__ __forceinline__ gv4f mfma4(float a, float b, gv4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ gv4f mfma_b(uint4 a, uint4 b, gv4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gb8, a), __builtin_bit_cast(gb8, b), c, 0, 0, 0);
}
// Product of operands of three parts in three independent chains, the small
// terms apart from hi hi. Left out: mid lo, lo mid, lo lo, below 2^-23 of hi hi
// and of either sign.
struct Acc3 {
    gv4f c[3] = {};
    __device__ __forceinline__ void add(const uint4 (&a)[3], const uint4 (&b)[3]) {
        c[0] = mfma_b(a[2], b[0], c[0]);
        c[1] = mfma_b(a[1], b[0], c[1]);
        c[2] = mfma_b(a[0], b[0], c[2]);
        c[0] = mfma_b(a[1], b[1], c[0]);
        c[1] = mfma_b(a[0], b[1], c[1]);
        c[0] = mfma_b(a[0], b[2], c[0]);
    }
    __device__ __forceinline__ gv4f sum() const { return (c[0] + c[1]) + c[2]; }
};

// Two values as three bf16 parts each: the high part cut off (no overflow), the
// rest rounded to the middle one, what is left exactly the low one. The values
// are rounded to fp32 first: a product folded into one use and not into another
// gives parts of different values.
__device__ __forceinline__ void split2(float x, float y, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
    asm("" : "+v"(x), "+v"(y));
    hi = __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u);
    x -= __uint_as_float(__float_as_uint(x) & 0xffff0000u);
    y -= __uint_as_float(__float_as_uint(y) & 0xffff0000u);
    mid = __builtin_bit_cast(uint32_t, (gb2){(__bf16)x, (__bf16)y});
    x -= __uint_as_float(mid << 16);
    y -= __uint_as_float(mid & 0xffff0000u);
    lo = __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u);
}
// A lane's fragment from two runs of four values.
__device__ __forceinline__ void split8(gv4f a, gv4f b, uint4 (&f)[3]) {
    split2(a[0], a[1], f[0].x, f[1].x, f[2].x);
    split2(a[2], a[3], f[0].y, f[1].y, f[2].y);
    split2(b[0], b[1], f[0].z, f[1].z, f[2].z);
    split2(b[2], b[3], f[0].w, f[1].w, f[2].w);
}
__device__ __forceinline__ void store3(uint4 *dst, const uint4 (&f)[3]) {
#pragma unroll
    for (int x = 0; x < 3; x++) dst[64 * x] = f[x];
}
__device__ __forceinline__ void load3(uint4 (&f)[3], const uint4 *src) {
#pragma unroll
    for (int x = 0; x < 3; x++) f[x] = src[64 * x];
}

// Sum over the four lane groups (lanes l, l ^ 16, l ^ 32).
__device__ __forceinline__ float groups_sum(float v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
}

// 16 x 16 tile of (rows of A) x (rows of B)^T over key_dim on fp32 MFMA: both
// operands in fragment order, a lane's 32 values of its row in 8 runs of four
// (run u at columns 16 u + 4 g). a: LDS row of lane m16, offset by 4 g.
__device__ __forceinline__ gv4f tile_rows(const float *a, const gv4f (&b)[8]) {
    // Four independent accumulation chains, summed at the end.
    gv4f c0 = {0.0f, 0.0f, 0.0f, 0.0f}, c1 = c0, c2 = c0, c3 = c0;
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const gv4f av = *(const gv4f *)(a + 16 * u);
        c0 = mfma4(av[0], b[u][0], c0);
        c1 = mfma4(av[1], b[u][1], c1);
        c2 = mfma4(av[2], b[u][2], c2);
        c3 = mfma4(av[3], b[u][3], c3);
    }
    return (c0 + c1) + (c2 + c3);
}

// Workgroup b runs on XCD b % 8. All workgroups of a head are placed on one
// XCD, so that they share the head's operands in that XCD's L2: XCD x takes
// heads x, x + 8, ..., `per` workgroups each (grid 8 * ceil(heads / 8) * per).
__device__ __forceinline__ void head_of_block(uint32_t block, uint32_t per, uint32_t &h, uint32_t &i) {
    const uint32_t q = block >> 3;
    h = (block & 7) + 8 * (q / per);
    i = q % per;
}

// Four values at columns col .. col + 3 of a row of `width` values (zeros past
// it, or all when !ok). VEC: width a multiple of 4 and the row 16-byte aligned;
// a compile-time choice, since a load behind a branch is waited for at its end.
template <bool VEC>
__device__ __forceinline__ gv4f load4(const float *row, uint32_t col, uint32_t width, bool ok) {
    gv4f r;
    if (VEC) {
        ok = ok && col < width;
        r = *(const gv4f *)(row + (ok ? col : 0));
#pragma unroll
        for (int x = 0; x < 4; x++) r[x] = ok ? r[x] : 0.0f;
    } else {
#pragma unroll
        for (int x = 0; x < 4; x++) r[x] = ok && col + x < width ? row[col + x] : 0.0f;
    }
    return r;
}

// Bound by issue and latency: one workgroup is a chain of about a dozen LDS
// exchanges around 320 fp32 MFMAs per wave (17.5 us alone on a CU, 13 us of the
// CU's time each when three share it; of 33000 clocks the loads take 8500, the
// tiles with A and L 10500, the inverse 9000, W and U 6000). K, Q and V are
// requested up front, Q stays in registers and V waits in them for K's LDS rows,
// T replaces L in place, so 52 KB of LDS let three workgroups share a CU.
template <bool VEC>
__device__ __forceinline__ void chunk_prep(const GdnArgs &a) {
    __shared__ __align__(16) float kh[GC * SPAD];  // raw K rows, then V rows
    __shared__ float tt[GC * TPAD];                // L, T, W's and then U's left operand
    __shared__ __align__(16) float G[GC], bt[GC], kinv_s[GC], ekf[GC];
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t m16 = lane & 15, g = lane >> 4;
    // On the XCD that reads the operands in pass 2: lines written on another one
    // cost both passes (us, this against heads in block order: 128 tokens of 32
    // heads 26.4 / 30.9, of 48 30.6 / 35.9, 320 of 32 34.3 / 35.4; 1280 and more
    // within 1%).
    uint32_t h, ci;
    head_of_block(blockIdx.x, a.chunks, h, ci);
    if (h >= a.heads) return;
    const uint32_t t0 = (a.chunk0 + ci) * a.chunk;
    const uint32_t n = min(a.chunk, a.tokens - t0);
    const uint32_t dk = a.key_dim, dv = a.value_dim;
    char *base = (char *)a.norms + ((size_t)h * a.chunks + ci) * CTOX_GDN_CHUNK_BYTES;
    float *aux = (float *)(base + GF_AUX);
    const float qscale = 1.0f / sqrtf((float)dk);
    const uint32_t own = 16 * w + m16;  // this lane's token of strip w

    const size_t th = (size_t)(t0 + min(lane, n - 1)) * a.heads + h;
    const float ld_raw = a.log_decay[th], bt_raw = a.beta[th];
    gv4f kr[8], qr[8], vr[8];
    {
        const size_t row = (size_t)(t0 + min(own, n - 1)) * a.qk_stride + (size_t)(h / a.rep) * dk;
#pragma unroll
        for (int u = 0; u < 8; u++) kr[u] = load4<VEC>(a.k + row, 16 * u + 4 * g, dk, own < n);
#pragma unroll
        for (int u = 0; u < 8; u++) qr[u] = load4<VEC>(a.q + row, 16 * u + 4 * g, dk, own < n);
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const uint32_t s = (tid >> 5) + 8 * u;
            vr[u] = load4<VEC>(a.v + (size_t)(t0 + min(s, n - 1)) * a.v_stride + (size_t)h * dv, (tid & 31) * 4, dv, s < n);
        }
    }
    // Inclusive prefix sum of log decay over the chunk (lane: token).
    float gl = lane < n ? ld_raw : 0.0f;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const float up = __shfl_up(gl, o);
        if (lane >= (uint32_t)o) gl += up;
    }
    const float gc = __shfl(gl, 63);
    if (w == 0) {
        G[lane] = gl;
        bt[lane] = lane < n ? bt_raw : 0.0f;
    }
    {
        float sq = 0.0f;
#pragma unroll
        for (int u = 0; u < 8; u++) {
            sq += (kr[u][0] * kr[u][0] + kr[u][1] * kr[u][1]) + (kr[u][2] * kr[u][2] + kr[u][3] * kr[u][3]);
            *(gv4f *)(kh + own * SPAD + 16 * u + 4 * g) = kr[u];
        }
        sq = groups_sum(sq);
        if (g == 0) kinv_s[own] = own < n ? 1.0f / sqrtf(sq + 1e-6f) : 0.0f;
    }
    float qinv;
    {   // Q fragments of strip w: normalised rows
        float sq = 0.0f;
#pragma unroll
        for (int u = 0; u < 8; u++)
            sq += (qr[u][0] * qr[u][0] + qr[u][1] * qr[u][1]) + (qr[u][2] * qr[u][2] + qr[u][3] * qr[u][3]);
        qinv = own < n ? 1.0f / sqrtf(groups_sum(sq) + 1e-6f) : 0.0f;
        uint4 *dst = (uint4 *)(base + GF_Q) + w * 768 + lane;
#pragma unroll
        for (int st = 0; st < 4; st++) {
            uint4 f[3];
            split8(qr[2 * st] * qinv, qr[2 * st + 1] * qinv, f);
            store3(dst + 192 * st, f);
        }
    }
    lds_barrier();
    if (w == 0) ekf[lane] = expf(gc - gl) * kinv_s[lane];
    // 16 x 16 tiles on the raw rows, scaled by the inverse norms afterwards,
    // five per wave: K Q^T of token strip w (rows r, columns t: the result is
    // A's fragment order) and K K^T of strip 3 - w.
    gv4f acc[5];
    const float *krow = kh + m16 * SPAD + 4 * g;
#pragma unroll
    for (uint32_t u = 0; u < 4; u++)
        if (u <= w) acc[u] = tile_rows(krow + 16 * u * SPAD, qr);
    {
        gv4f ks[8];  // strip 3 - w as the right operand
#pragma unroll
        for (int u = 0; u < 8; u++) ks[u] = *(const gv4f *)(krow + 16 * (3 - w) * SPAD + 16 * u);
#pragma unroll
        for (uint32_t u = 1; u < 5; u++)
            if (u > w) acc[u] = tile_rows(krow + 16 * (u - w - 1) * SPAD, ks);
    }
    {   // A: row t = own, this lane's r = 16 u + 4 g + x
        const float Gown = G[own];
#pragma unroll
        for (uint32_t u = 0; u < 4; u++) {
            if (u > w) continue;
            const gv4f Gr = *(const gv4f *)&G[16 * u + 4 * g], kr4 = *(const gv4f *)&kinv_s[16 * u + 4 * g];
#pragma unroll
            for (int x = 0; x < 4; x++) {
                const uint32_t r = 16 * u + 4 * g + x;
                acc[u][x] = r <= own ? expf(Gown - Gr[x]) * (kr4[x] * qinv) * acc[u][x] : 0.0f;
            }
        }
        uint4 *dst = (uint4 *)(base + GF_A) + w * 384 + lane;
        const gv4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
        uint4 f[3];
        split8(acc[0], w >= 1 ? acc[1] : zero, f);
        store3(dst, f);
        split8(w >= 2 ? acc[2] : zero, w >= 3 ? acc[3] : zero, f);
        store3(dst + 192, f);
    }
    {   // L of strip 3 - w, strictly lower: the tile's rows are r, its columns s
        const uint32_t s = 16 * (3 - w) + m16;
        const float f = bt[s] * kinv_s[s], Gs = G[s];
#pragma unroll
        for (uint32_t u = 1; u < 5; u++) {
            if (u <= w) continue;
            const gv4f kr4 = *(const gv4f *)&kinv_s[16 * (u - w - 1) + 4 * g], Gr = *(const gv4f *)&G[16 * (u - w - 1) + 4 * g];
#pragma unroll
            for (int x = 0; x < 4; x++) {
                const uint32_t r = 16 * (u - w - 1) + 4 * g + x;
                tt[s * TPAD + r] = r < s ? expf(Gs - Gr[x]) * (f * kr4[x]) * acc[u][x] : 0.0f;
            }
        }
    }
    lds_barrier();
    // T = (I + L)^{-1} over L, blockwise over 16 x 16 blocks:
    //   T_ii = (I + L_ii)^{-1}                   forward substitution, wave i
    //                                            (row s of L is last read for row s of T);
    //   T_ij = -T_ii sum_{k=j}^{i-1} L_ik T_kj   block row i after row i - 1,
    //                                            task j on wave j, on MFMA.
    if (lane < 16) {
        float *blk = tt + 16 * w * TPAD + 16 * w;
        float col[16];
#pragma unroll
        for (int s = 0; s < 16; s++) {
            float sum = 0.0f;
#pragma unroll
            for (int r = 0; r < s; r++) sum = fmaf(blk[s * TPAD + r], col[r], sum);
            col[s] = ((uint32_t)s == lane ? 1.0f : 0.0f) - sum;
        }
#pragma unroll
        for (int s = 0; s < 16; s++) blk[s * TPAD + lane] = col[s];
    }
    {   // K^T fragments of key tiles 2 w, 2 w + 1, with the decay to the chunk's end
        uint4 *dst = (uint4 *)(base + GF_K) + w * 768 + lane;
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const float *kp = kh + 16 * (2 * w + t) + m16;
#pragma unroll
            for (int st = 0; st < 2; st++) {
                gv4f lo = *(const gv4f *)&ekf[32 * st + 4 * g], up = *(const gv4f *)&ekf[32 * st + 16 + 4 * g];
#pragma unroll
                for (int x = 0; x < 4; x++) {
                    const uint32_t r = 32 * st + 4 * g + x;
                    lo[x] *= kp[r * SPAD];
                    up[x] *= kp[(r + 16) * SPAD];
                }
                uint4 f[3];
                split8(lo, up, f);
                store3(dst + 384 * t + 192 * st, f);
            }
        }
    }
#pragma unroll
    for (uint32_t bi = 1; bi < 4; bi++) {
        lds_barrier();  // block row bi - 1 (and the diagonal) written
        // X = sum_k L_ik T_kj: A = L rows of block bi, B = T rows of block k.
        gv4f y = {0.0f, 0.0f, 0.0f, 0.0f};
        if (w < bi) {
            gv4f x = y;
            for (uint32_t bk = w; bk < bi; bk++) {
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    const uint32_t kk = 16 * bk + 4 * u + g;
                    x = mfma4(tt[(16 * bi + m16) * TPAD + kk], tt[kk * TPAD + 16 * w + m16], x);
                }
            }
            // T_ij = -T_ii X. Lane (g, n) holds X rows 4 g + u of column n, so
            // MFMA u takes k = 4 g + u: A reads T_ii[m][4 g + u].
#pragma unroll
            for (int u = 0; u < 4; u++) y = mfma4(tt[(16 * bi + m16) * TPAD + 16 * bi + 4 * g + u], x[u], y);
        }
        lds_barrier();  // block row bi of L is dead
        if (w < bi) {
#pragma unroll
            for (int u = 0; u < 4; u++) tt[(16 * bi + 4 * g + u) * TPAD + 16 * w + m16] = -y[u];
        }
    }
    lds_barrier();
    // tt: T diag(b g kinv) (W's left operand, on the raw K rows); in registers,
    // for tt later: T diag(b) (U's). Lane: column r, rows 16 w + i.
    // Blocks above the diagonal are read by no product.
    float tu[16];
    {
        const float b = bt[lane], ki = kinv_s[lane] * expf(gl);
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const uint32_t s = 16 * w + i;
            const float t = tt[s * TPAD + lane] * b;
            tu[i] = t;
            tt[s * TPAD + lane] = t * ki;
        }
    }
    lds_barrier();
    // W^T of key tiles 2 w, 2 w + 1 (rows i, columns s: W's fragment order).
    gv4f wt[4][2];
#pragma unroll
    for (int st = 0; st < 4; st++) wt[st][0] = wt[st][1] = gv4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int rb = 0; rb < 4; rb++)
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint32_t r = 16 * rb + 4 * u + g;
            const float a0 = kh[r * SPAD + 32 * w + m16], a1 = kh[r * SPAD + 32 * w + 16 + m16];
#pragma unroll
            for (int st = rb; st < 4; st++) {
                const float b = tt[(16 * st + m16) * TPAD + r];
                wt[st][0] = mfma4(a0, b, wt[st][0]);
                wt[st][1] = mfma4(a1, b, wt[st][1]);
            }
        }
    lds_barrier();  // K rows and W's left operand are dead
#pragma unroll
    for (int i = 0; i < 16; i++) tt[(16 * w + i) * TPAD + lane] = tu[i];
#pragma unroll
    for (int u = 0; u < 8; u++) *(gv4f *)(kh + ((tid >> 5) + 8 * u) * SPAD + (tid & 31) * 4) = vr[u];
    {
        uint4 *dst = (uint4 *)(base + GF_W) + 192 * w + lane;
#pragma unroll
        for (int st = 0; st < 4; st++) {
            uint4 f[3];
            split8(wt[st][0], wt[st][1], f);
            store3(dst + 768 * st, f);
        }
    }
    if (w == 0) {
        const float ge = expf(gl);
        aux[lane] = qscale * ge;
        if (lane == GC - 1) aux[64] = ge;
    }
    lds_barrier();
    // U of value tiles 2 w, 2 w + 1.
    if (32 * w >= dv) return;
    gv4f us[4][2];
#pragma unroll
    for (int st = 0; st < 4; st++) us[st][0] = us[st][1] = gv4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int rb = 0; rb < 4; rb++)
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint32_t r = 16 * rb + 4 * u + g;
            const float v0 = kh[r * SPAD + 32 * w + m16], v1 = kh[r * SPAD + 32 * w + 16 + m16];
#pragma unroll
            for (int st = rb; st < 4; st++) {
                const float t = tt[(16 * st + m16) * TPAD + r];
                us[st][0] = mfma4(t, v0, us[st][0]);
                us[st][1] = mfma4(t, v1, us[st][1]);
            }
        }
    float4 *dst = (float4 *)(base + GF_U) + 512 * w + lane;
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const gv4f x = us[st][j];
            dst[256 * j + 64 * st] = make_float4(x[0], x[1], x[2], x[3]);
        }
}

// A chunk's operands of one wave, in registers one chunk ahead.
template <int NT>
struct GdnStateOps {     // waves 0..3
    uint4 w[4][3];       // W strip, key steps
    uint4 k[2][2][3];    // K^T key tiles 2 w, 2 w + 1, token steps
    float4 u[NT];
    float gc;
};
struct GdnOutOps {       // waves 4..7
    uint4 q[4][3];
    uint4 am[2][3];
    float4 fq;
};

// The operands' exchange. One buffer each: state operands are read between the
// first barrier of a chunk and its second, D's after it.
template <int NT>
struct GdnScanLds {
    uint4 s[NT][4][3][64];    // [value tile][key step][part][lane]
    uint4 d[NT][2][3][64];    // [value tile][token step][part][lane]; a strip is half of each 16 B
};

// X = (rows) x S_0. fetch(k) issues a quarter of the next chunk's loads.
template <int NT, class Fetch>
__device__ __forceinline__ gv4f times_state(const uint4 (&x)[4][3], const GdnScanLds<NT> &L, int j, uint32_t lane,
                                            Fetch fetch) {
    Acc3 acc;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        fetch(k);
        __builtin_amdgcn_sched_barrier(0);
        const uint4 s[3] = {L.s[j][k][0][lane], L.s[j][k][1][lane], L.s[j][k][2][lane]};
        acc.add(x[k], s);
    }
    return acc.sum();
}

// NT: value tiles (of 16 columns) per workgroup.
template <int NT>
__device__ __forceinline__ void chunk_scan(const GdnArgs &a) {
    __shared__ GdnScanLds<NT> L;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t m16 = lane & 15, g = lane >> 4, w = wave & 3;
    const uint32_t slices = (a.value_dim + 16 * NT - 1) / (16 * NT);
    uint32_t h, slice;
    head_of_block(blockIdx.x, slices, h, slice);
    if (h >= a.heads) return;
    const uint32_t dk = a.key_dim, dv = a.value_dim, nch = a.chunks, j0 = slice * 16 * NT;
    const char *scratch = (const char *)a.norms + (size_t)h * nch * CTOX_GDN_CHUNK_BYTES;
    const bool second = a.chunk > 32;  // tokens in the second step

    if (wave < 4) {
        // part 0..3: W of a key step (and the small operands), 4: K^T of the first key tile, 5: of the second.
        auto load = [&](GdnStateOps<NT> &p, uint32_t c, int part) {
            const char *b = scratch + (size_t)min(c, nch - 1) * CTOX_GDN_CHUNK_BYTES;
            const uint4 *wp = (const uint4 *)(b + GF_W) + 768 * w + lane, *kp = (const uint4 *)(b + GF_K) + 768 * w + lane;
            const float4 *up = (const float4 *)(b + GF_U) + 256 * (NT * slice) + 64 * w + lane;
            if (part < 4) load3(p.w[part], wp + 192 * part);
            if (part == 0) p.gc = ((const float *)(b + GF_AUX))[64];
            if (part == 1) {
#pragma unroll
                for (int j = 0; j < NT; j++) p.u[j] = up[256 * j];
            }
            if (part >= 4) {
#pragma unroll
                for (int u = 0; u < 2; u++) load3(p.k[part - 4][u], kp + 384 * (part - 4) + 192 * u);
            }
        };
        // State rows 32 w + 16 t + 4 g + r, column j0 + 16 j + m16.
        gv4f st[NT][2];
        float *S = a.state + (size_t)h * dk * dv;
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    // (no branch around the load: they are all in flight at once)
                    const uint32_t i = 32 * w + 16 * t + 4 * g + r, col = j0 + 16 * j + m16;
                    const float x = S[(size_t)min(i, dk - 1) * dv + min(col, dv - 1)];
                    st[j][t][r] = i < dk && col < dv ? x : 0.0f;
                }
        auto publish = [&](int j) {
            uint4 f[3];
            split8(st[j][0], st[j][1], f);
            store3(&L.s[j][w][0][lane], f);
        };
        auto step = [&](const GdnStateOps<NT> &p, GdnStateOps<NT> &nx, uint32_t c) {
#pragma unroll
            for (int j = 0; j < NT; j++) {
                const gv4f x = times_state<NT>(p.w, L, j, lane, [&](int k) {
                    if (j == 0) load(nx, c + 1, k);
                });
                uint2 f[3];
                split2(p.u[j].x - x[0], p.u[j].y - x[1], f[0].x, f[1].x, f[2].x);
                split2(p.u[j].z - x[2], p.u[j].w - x[3], f[0].y, f[1].y, f[2].y);
#pragma unroll
                for (int i = 0; i < 3; i++) ((uint2 *)&L.d[j][w >> 1][i][lane])[w & 1] = f[i];
            }
            lds_barrier();
#pragma unroll
            for (int j = 0; j < NT; j++) {
                if (j == 0) load(nx, c + 1, 4);
                Acc3 n0, n1;
                const uint4 d0[3] = {L.d[j][0][0][lane], L.d[j][0][1][lane], L.d[j][0][2][lane]};
                n0.add(p.k[0][0], d0);
                n1.add(p.k[1][0], d0);
                if (second) {
                    const uint4 d1[3] = {L.d[j][1][0][lane], L.d[j][1][1][lane], L.d[j][1][2][lane]};
                    n0.add(p.k[0][1], d1);
                    n1.add(p.k[1][1], d1);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (j == 0) load(nx, c + 1, 5);
                st[j][0] = st[j][0] * p.gc + n0.sum();
                st[j][1] = st[j][1] * p.gc + n1.sum();
                publish(j);
            }
            lds_barrier();
        };
        GdnStateOps<NT> pa, pb;
#pragma unroll
        for (int part = 0; part < 6; part++) load(pa, 0, part);
#pragma unroll
        for (int j = 0; j < NT; j++) publish(j);
        lds_barrier();
        for (uint32_t c = 0; c < nch; c += 2) {
            step(pa, pb, c);
            if (c + 1 == nch) break;
            step(pb, pa, c + 1);
        }
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const uint32_t i = 32 * w + 16 * t + 4 * g + r, col = j0 + 16 * j + m16;
                    if (i < dk && col < dv) S[(size_t)i * dv + col] = st[j][t][r];
                }
    } else {
        // part 0..3: Q of a key step (and the small operands), 4, 5: A of a token step.
        auto load = [&](GdnOutOps &p, uint32_t c, int part) {
            const char *b = scratch + (size_t)min(c, nch - 1) * CTOX_GDN_CHUNK_BYTES;
            const uint4 *qp = (const uint4 *)(b + GF_Q) + 768 * w + lane, *ap = (const uint4 *)(b + GF_A) + 384 * w + lane;
            if (part < 4) load3(p.q[part], qp + 192 * part);
            if (part == 1) p.fq = *(const float4 *)((const float *)(b + GF_AUX) + 16 * w + 4 * g);
            if (part >= 4) load3(p.am[part - 4], ap + 192 * (part - 4));
        };
        const size_t rowv = (size_t)a.heads * dv;
        const float qscale = 1.0f / sqrtf((float)dk);
        auto step = [&](const GdnOutOps &p, GdnOutOps &nx, uint32_t c) {
            gv4f o[NT];
#pragma unroll
            for (int j = 0; j < NT; j++)
                o[j] = times_state<NT>(p.q, L, j, lane, [&](int k) {
                    if (j == 0) load(nx, c + 1, k);
                });
            lds_barrier();
            load(nx, c + 1, 4);
            load(nx, c + 1, 5);
            const uint32_t t0 = (a.chunk0 + c) * a.chunk, n = min(a.chunk, a.tokens - t0);
            float *out = a.out + (size_t)t0 * rowv + (size_t)h * dv + j0 + m16;
#pragma unroll
            for (int j = 0; j < NT; j++) {
                Acc3 acc;
                const uint4 d0[3] = {L.d[j][0][0][lane], L.d[j][0][1][lane], L.d[j][0][2][lane]};
                acc.add(p.am[0], d0);
                if (w >= 2 && second) {  // strips 0 and 1 see no token of the second step
                    const uint4 d1[3] = {L.d[j][1][0][lane], L.d[j][1][1][lane], L.d[j][1][2][lane]};
                    acc.add(p.am[1], d1);
                }
                const gv4f x = acc.sum();
                const float fq[4] = {p.fq.x, p.fq.y, p.fq.z, p.fq.w};
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const uint32_t s = 16 * w + 4 * g + r;
                    if (s < n && j0 + 16 * j + m16 < dv) out[(size_t)s * rowv + 16 * j] = fq[r] * o[j][r] + qscale * x[r];
                }
            }
            lds_barrier();
        };
        GdnOutOps pa, pb;
#pragma unroll
        for (int part = 0; part < 6; part++) load(pa, 0, part);
        lds_barrier();
        for (uint32_t c = 0; c < nch; c += 2) {
            step(pa, pb, c);
            if (c + 1 == nch) break;
            step(pb, pa, c + 1);
        }
    }
}

// _vec: key_dim, value_dim and the token strides are multiples of 4 and q, k, v 16-byte aligned.
extern "C" __global__ __launch_bounds__(256, 3) void ctox_gdn_chunk_prep_gfx950(GdnArgs a) { chunk_prep<false>(a); }
extern "C" __global__ __launch_bounds__(256, 3) void ctox_gdn_chunk_prep_vec_gfx950(GdnArgs a) { chunk_prep<true>(a); }
extern "C" __global__ __launch_bounds__(512) void ctox_gdn_chunk_scan1_gfx950(GdnArgs a) { chunk_scan<1>(a); }
extern "C" __global__ __launch_bounds__(512) void ctox_gdn_chunk_scan2_gfx950(GdnArgs a) { chunk_scan<2>(a); }
