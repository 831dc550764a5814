/* Quantized GEMM on the matrix cores for every supported type (gfx950):
 *     Y[t, r] = W[r, :] . X[t, :],  t < M tokens, r < N rows, K = cols.
 *
 * Replaces the int8 MMA kernels mmq*_<ty> / mmq128r_<ty> behind DenseGpu::bmm and prefill::dense
 * (src/cuda/kernels.cu:965-1235, src/gpu/dense.rs:181-199, src/gpu/prefill.rs:44-60); CPU twin
 * cpu_ref::matmat (src/cpu_ref.rs:266-276).
 *
 * Operands. v_mfma_f32_32x32x16_f16 with the tokens as A (32 x 16) and the weight rows as B
 * (16 x 32), fp32 accumulation. Lane l of a fragment holds token / row l % 32 and the eight K
 * positions 8 (l / 32) .. +8 of the 16-value K chunk, stored in the order P8 = 0,2,1,3,4,6,5,7
 * (what the byte-pair fp16 conversion below produces; the dot product does not depend on the
 * order as long as A and B agree).
 *
 * Activations (pre-pass le_gq_xprep_*). Token t is scaled by 2^-e_t, e_t chosen so that
 * max|x_t| 2^-e_t lies in [64, 128) (exact: a power of two), and rounded to fp16 (relative error
 * 2^-11; values below 2^-24 of the token's maximum flush towards zero). The result is written in
 * fragment order, [32-token tile][K/16 chunk][8-lane half][token][8 halves], so a block copies
 * each step's activations as contiguous 8 KB runs and every A fragment is one conflict-free
 * 16-byte LDS read per lane. Q4_K and Q5_K also get per-super-block sub-block sums S_j (per 32
 * values, as fp16 high + low halves) for their offset term. The final store multiplies by
 * 2^e_t, so the result does not depend on the activations' magnitude.
 *
 * Weights. Raw GGUF rows (src/gpu.rs:79-83), read in half super-blocks (128 values) per pipeline
 * step: each row's bytes for the step are copied as 16-byte chunks (coalesced: consecutive lanes
 * take consecutive chunks of a row) into a 16-byte-aligned LDS slot of F::SLOT bytes, then each
 * lane builds its B fragments from them:
 *   Q4_K   code sc_j * q (<= 945, exact), offset term D2 = sum_j m_j S_j (one more MFMA per
 *          super-block), acc = acc (d' / d) + D1 - (dmin / d) D2, in units of d    (src/quant.rs:72-82)
 *   Q6_K   code (q6 - 32) * sc_u / 64 (exact where (q6 - 32) sc_u has at most 11 significant
 *          bits, else rounded once to fp16), scale 64 d                          (:96-112)
 *   IQ2_XXS code (2s+1) * grid * sign (<= 1333, exact), scale d/8                  (:142-154)
 *   IQ3_XXS code (2s+1) * grid * sign (<= 1922, exact), scale d/4                  (:127-141)
 *   Q5_K   as Q4_K with the fifth bit from qh, code sc_j * q (<= 1953, exact)     (:83-95)
 *   Q3_K   code (q3 - 4) * (sc6 - 32) (|.| <= 128, exact), scale d                (:113-126)
 *   IQ2_S  code (2s+1) * grid * sign, 1024-entry grid, explicit sign bytes, scale d/8
 *                                                                                  (:155-167)
 *   Q8_0, Q4_0  per-32 scale d_b inside the code: fp16(q * d_b 2^S) (one rounding, 2^-11
 *          relative), S a per-row power of two that only decreases (the accumulator is rescaled
 *          when it does) and keeps every code inside the fp16 range, final * 2^-S  (:64-71)
 * A scale: acc = acc (previous scale / scale) + D1, the accumulator in units of the row's last scale.
 * Integer byte -> fp16 conversion: a byte u placed under the fp16 exponent of 1024 (v_perm_b32)
 * is the half 1024 + u exactly; one packed fma (u+1024)*c - 1024*c gives u*c rounded once.
 *
 * Tiling. A block of WM x WN waves computes BM = 32 TM WM tokens x BN = 32 TN WN rows; a wave
 * owns TM x TN 32x32 tiles. Steps are double-buffered in LDS; every thread holds two further
 * steps of loads in registers (issued two steps before they are written to LDS), so the loads of
 * steps s+2 and s+3 are in flight while step s computes. Blocks that share weight rows (same row
 * tile, other token tiles or K slices) get the same blockIdx % 8 and therefore the same XCD and
 * L2. With fewer than 8 row tiles, row tiles vary fastest instead, so the blocks
 * spread over all XCDs. K may be split over blockIdx.y; the slices' partial results are then
 * summed by le_gq_ksum (or, without room for them, added into Y atomically after the pre-pass
 * cleared it).
 */
#include "le_f16_frag.h"

struct GqArgs {
    const u8 *w;
    const float *x;
    float *y;
    int rows, cols, m;
    int mp;     /* tokens rounded up to the largest token tile (the pre-pass pads with zeros) */
    int ksplit; /* K slices (blockIdx.y); > 1: partial sums into part (then le_gq_ksum), or, with no
                 * part buffer, atomic adds into y, cleared by the pre-pass */
    /* grouped form (le_mm_grouped): slot s multiplies weight ptrs[s] (or w + s * w_slot_bytes)
     * with the activation rows in_idx[i] of its pairs i in off[s] .. off[s+1], writing output rows
     * out_idx[i]; the plan kernel lists (slot, first pair) token tiles of bm pairs in the workspace */
    const u8 *const *ptrs;
    unsigned long long w_slot_bytes;
    const int *off, *in_idx, *out_idx;
    int nslot, maxt, bm, npair; /* grouped form: npair pairs (the pre-pass's grid) */
    float *part; /* [ksplit][m][rows] partial results of the K slices, or null */
    /* grouped form, dual: a second weight set (ptrs2 or w2, same type and shape) applied to the same
     * pairs, written to y2 (the MoE gate and up projections in one launch) */
    const u8 *const *ptrs2;
    const u8 *w2;
    float *y2;
    int dual, ids; /* ids: blocks of the whole grouped launch (le_gqu_*) */
    const float *up; /* non-null: the activation rows are silu(x) * up (the MoE down input) */
};

/* Workspace layout: A planes (mp * K halves), S records (mp/32 * nsb * SREC bytes), token scales
 * (mp floats). */
__host__ __device__ inline size_t gq_s_off(int mp, int K) { return (size_t)mp * K * 2; }
__host__ __device__ inline size_t gq_t_off(int mp, int K, int srec) { return gq_s_off(mp, K) + (size_t)(mp / 32) * (K / 256) * srec; }

__device__ __forceinline__ void gq_barrier() {
    __asm__ volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F); /* LDS only: the loads of later steps stay in flight */
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
}

template <int TM, int TN>
__device__ __forceinline__ void gq_mma(le_v16f (&d)[TM][TN], const le_v8h (&A)[TM], const le_v8h (&B)[TN], bool zero) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int k = 0; k < TN; k++) d[i][k] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[i], B[k], zero ? (le_v16f){} : d[i][k], 0, 0, 0);
}

/* ============================ per-type formats ============================
 * SBB: bytes per super-block; NCH 16-byte chunks per row and step, chunk k of half h read from
 * byte goff(k, h) of the super-block into byte loff(k) of the row's slot; SREC: bytes of sum
 * records per (32-token tile, super-block); EPI: 1 if the per-super-block epilogue is used. */
template <int TY>
struct GqF;

template <>
struct GqF<LE_TYPE_Q4_K> { /* slot: [0,16) header, [16,80) this half's 64 quant bytes */
    static constexpr int SBB = 144, NCH = 5, SLOT = 80, SREC = 1024, EPI = 1, TAB = 0;
    static constexpr bool ALIGNED = true;
    __device__ static int goff(int k, int h) { return k == 0 ? 0 : 16 + 64 * h + 16 * (k - 1); }
    __device__ static float scale(const u8 *r) { return h2f(*(const uint16_t *)r); }
    __device__ static int loff(int k) { return 16 * k; }
};
template <>
struct GqF<LE_TYPE_Q6_K> { /* slot: [0,64) ql half, [64,96) qh half, [96,112) sc[16], [112,128) bytes 194..209 (d at 126);
                             * 144-byte stride: at 128 the 32 rows of a fragment read fell into two bank groups */
    static constexpr int SBB = 210, NCH = 8, SLOT = 144, SREC = 0, EPI = 1, TAB = 0;
    static constexpr bool ALIGNED = false;
    __device__ static int goff(int k, int h) {
        return k < 4 ? 64 * h + 16 * k : k < 6 ? 128 + 32 * h + 16 * (k - 4) : k == 6 ? 192 : 194;
    }
    __device__ static float scale(const u8 *r) { return 64.f * h2f(*(const uint16_t *)(r + 126)); }
    __device__ static int loff(int k) { return 16 * k; }
};
template <>
struct GqF<LE_TYPE_Q5_K> { /* slot: [0,16) header, [16,48) qh (all 32 bytes), [48,112) this half's 64 quant bytes */
    static constexpr int SBB = 176, NCH = 7, SLOT = 112, SREC = 1024, EPI = 1, TAB = 0;
    static constexpr bool ALIGNED = true;
    __device__ static int goff(int k, int h) { return k < 3 ? 16 * k : 48 + 64 * h + 16 * (k - 3); }
    __device__ static float scale(const u8 *r) { return h2f(*(const uint16_t *)r); }
    __device__ static int loff(int k) { return 16 * k; }
};
template <>
struct GqF<LE_TYPE_Q3_K> { /* slot: [0,32) the half's 32 quant bytes, [32,64) hmask, [64,80) bytes 94..109 (scales at
                             * 66..77, d at 78) */
    static constexpr int SBB = 110, NCH = 5, SLOT = 80, SREC = 0, EPI = 1, TAB = 0;
    static constexpr bool ALIGNED = false;
    __device__ static int goff(int k, int h) { return k < 2 ? 32 + 32 * h + 16 * k : k < 4 ? 16 * (k - 2) : 94; }
    __device__ static float scale(const u8 *r) { return h2f(*(const uint16_t *)(r + 78)); }
    __device__ static int loff(int k) { return 16 * k; }
};
template <>
struct GqF<LE_TYPE_IQ2_S> { /* slot: [0,16) the half's grid index bytes, [16,32) its sign bytes, [32,48) bytes 66..81
                             * (qh[8], scales[8]), [48,64) bytes 0..15 (d at 48) */
    static constexpr int SBB = 82, NCH = 4, SLOT = 80, SREC = 0, EPI = 1, TAB = 16384 + 4096;
    static constexpr bool ALIGNED = false;
    __device__ static int goff(int k, int h) { return k == 0 ? 2 + 16 * h : k == 1 ? 34 + 16 * h : k == 2 ? 66 : 0; }
    __device__ static float scale(const u8 *r) { return 0.125f * h2f(*(const uint16_t *)(r + 48)); }
    __device__ static int loff(int k) { return 16 * k; }
};
template <>
struct GqF<LE_TYPE_Q4_0> { /* 8 blocks of 18 bytes form a 144-byte super-block; slot: [16b, 16b+16) quant bytes of block b
                            * of the half, [64 + 16b] chunk starting at d_b; 144-byte stride */
    static constexpr int SBB = 144, NCH = 8, SLOT = 144, SREC = 0, EPI = 2, TAB = 0;
    static constexpr bool ALIGNED = false;
    __device__ static int goff(int k, int h) { return k < 4 ? 72 * h + 18 * k + 2 : 72 * h + 18 * (k - 4); }
    __device__ static float scale(const u8 *r) { return 1.f; }
    __device__ static int loff(int k) { return 16 * k; }
};
template <>
struct GqF<LE_TYPE_Q8_0> { /* slot: [32b, 32b+32) quants of block b of the half, [128 + 16b] chunk starting at d_b */
    static constexpr int SBB = 272, NCH = 12, SLOT = 192, SREC = 0, EPI = 2, TAB = 0;
    static constexpr bool ALIGNED = false;
    __device__ static int goff(int k, int h) {
        return k < 8 ? 136 * h + 34 * (k >> 1) + 2 + 16 * (k & 1) : 136 * h + 34 * (k - 8);
    }
    __device__ static float scale(const u8 *r) { return 1.f; }
    __device__ static int loff(int k) { return 16 * k; }
};
template <>
struct GqF<LE_TYPE_IQ2_XXS> { /* slot: [0,32) the half's four 8-byte block records, [32,48) bytes 0..15 (d at 32) */
    static constexpr int SBB = 66, NCH = 3, SLOT = 48, SREC = 0, EPI = 1, TAB = 4096 + 2048;
    static constexpr bool ALIGNED = false;
    __device__ static int goff(int k, int h) { return k < 2 ? 2 + 32 * h + 16 * k : 0; }
    __device__ static float scale(const u8 *r) { return 0.125f * h2f(*(const uint16_t *)(r + 32)); }
    __device__ static int loff(int k) { return 16 * k; }
};
template <>
struct GqF<LE_TYPE_IQ3_XXS> { /* slot: [0,32) the half's grid indices, [32,48) its four aux words, [48,64) bytes 0..15 (d at 48);
                                * 80-byte stride, as Q6_K's */
    static constexpr int SBB = 98, NCH = 4, SLOT = 80, SREC = 0, EPI = 1, TAB = 2048 + 2048;
    static constexpr bool ALIGNED = false;
    __device__ static int goff(int k, int h) { return k < 2 ? 2 + 32 * h + 16 * k : k == 2 ? 66 + 16 * h : 0; }
    __device__ static float scale(const u8 *r) { return 0.25f * h2f(*(const uint16_t *)(r + 48)); }
    __device__ static int loff(int k) { return 16 * k; }
};

/* ============================ activation pre-pass ============================ */
/* pre-pass: group g (8 values 8g..8g+7 = chunk g / 2, half g & 1) of padded token t, scaled by sc,
 * into the fp16 fragments A and (SK) the sum records S. The 2 or 4 lanes of one sum are g's
 * neighbours in the same wave, all inside or all outside the row (K % 256 == 0). */
template <int SK>
__device__ __forceinline__ void gq_xconvert(int g, float4 p, float4 q, float sc, int t, int K, _Float16 *A, u8 *S) {
    constexpr int SREC = SK == 1 ? 1024 : 2048;
    const int nsb = K >> 8, tile = t >> 5, tl = t & 31;
    float v[8] = {p.x * sc, p.y * sc, p.z * sc, p.w * sc, q.x * sc, q.y * sc, q.z * sc, q.w * sc};
    const le_h2 h0 = {(_Float16)v[0], (_Float16)v[2]}, h1 = {(_Float16)v[1], (_Float16)v[3]};
    const le_h2 h2 = {(_Float16)v[4], (_Float16)v[6]}, h3 = {(_Float16)v[5], (_Float16)v[7]};
    const size_t off = ((((size_t)tile * (K / 16) + (g >> 1)) * 2 + (g & 1)) * 32 + tl) * 8;
    *(LE_GLOBAL uint4 *)(A + off) = make_uint4(as_u32(h0), as_u32(h1), as_u32(h2), as_u32(h3));
    if constexpr (SK != 0) {
        /* g runs over consecutive lanes, so the groups of one sum are neighbouring lanes */
        /* sums of the fp16-rounded values the MFMA sees, so that the mins term cancels the
         * scale term's share of the rounding exactly: the result is then sum w * x~ with
         * error relative to sum |w x|, not to sum |sc q x| */
        float r[8];
#pragma unroll
        for (int i = 0; i < 8; i++) r[i] = (float)(_Float16)v[i];
        float s = ((r[0] + r[1]) + (r[2] + r[3])) + ((r[4] + r[5]) + (r[6] + r[7]));
        s += __shfl_xor(s, 1);
        if constexpr (SK == 1) s += __shfl_xor(s, 2);
        const int span = SK == 1 ? 4 : 2;
        if ((g & (span - 1)) == 0) {
            const int sb = g >> 5, j = (g & 31) / span; /* sum index within the super-block */
            const _Float16 hi = (_Float16)s, lo = (_Float16)(s - (float)hi);
            _Float16 *rec = (_Float16 *)(S + ((size_t)tile * nsb + sb) * SREC);
            /* position P8(j % 8) (P8 is its own inverse), the order of the B2 operand */
            const int pj = (j & 4) | ((j & 1) << 1) | ((j >> 1) & 1);
            if constexpr (SK == 1) { /* [hs][token][8]: hs 0 high halves, hs 1 low halves */
                rec[tl * 8 + pj] = hi;
                rec[256 + tl * 8 + pj] = lo;
            } else { /* [f][hs][token][8]: f 0 high, f 1 low; hs = j / 8 */
                rec[((j >> 3) * 32 + tl) * 8 + pj] = hi;
                rec[512 + ((j >> 3) * 32 + tl) * 8 + pj] = lo;
            }
        }
    }
}


/* One block of 256 threads per (padded) token, or per pair in the grouped form. SK: 0 no sums, 1 per-32 sums (Q4_K), 2 per-16
 * sums (Q6_K). */
template <int SK, bool GR = false>
__device__ __forceinline__ void gq_xprep_body(const GqArgs &a, u8 *ws) {
    __shared__ float red[4];
    const int K = a.cols, nsb = K >> 8, tid = threadIdx.x, lane = tid & 63;
    int t = blockIdx.x; /* padded token (grouped form: the pair's tile position, below) */
    if (!GR && a.ksplit > 1 && !a.part) { /* the slices add into y */
        const size_t ny = (size_t)a.m * a.rows, st = (size_t)gridDim.x * blockDim.x;
        size_t i = (size_t)blockIdx.x * blockDim.x + tid;
        if ((ny & 3) == 0 && ((size_t)a.y & 15) == 0)
            for (; i < ny / 4; i += st) ((float4 *)a.y)[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        else
            for (; i < ny; i += st) a.y[i] = 0.f;
    }
    bool live = t < a.m;
    size_t src = t;
    if constexpr (GR) {
        /* one block per pair p (the grid is npair blocks): its slot s (off[s] <= p < off[s+1]),
         * then its position first_tile(s) * bm + (p - off[s]) among the tiles; the pair's token
         * index loads with the slots' offsets */
        const int p = blockIdx.x;
        const int srcp = a.in_idx[p];
        live = false;
        int o0, first;
        const int lo = le_slot_walk(a.off, a.nslot, a.bm, [p](int b, int e, int, int) { return p >= b && p < e; }, o0, first);
        if (lo >= 0) {
            const int j = p - o0, tile = first + j / a.bm;
            if (tile < a.maxt) {
                live = true;
                t = tile * a.bm + j % a.bm;
                src = (size_t)srcp;
            }
        }
    }
    /* grouped form: a tile position without a pair writes nothing. Its activation rows, sums and
     * scale are never combined with a valid row (an MFMA output row depends on its own A row
     * only) and its outputs are not stored, so whatever the workspace holds there is harmless. */
    if (GR && !live) return;
    const LE_GLOBAL float *xr = (const LE_GLOBAL float *)(a.x + (live ? src : 0) * K);
    /* up to K = 16384 every thread keeps its groups' values in registers between the max and the
     * conversion: one read of the token, all of a thread's loads in flight at once */
    constexpr int XG = 8;
    const int ng = K / 8;
    const bool inreg = ng <= 256 * XG;
    float4 P[XG], Q[XG];
    float am = 0.f;
    if (inreg) {
#pragma unroll
        for (int i = 0; i < XG; i++) {
            const int g = tid + 256 * i;
            if (live && g < ng) {
                P[i] = ((const LE_GLOBAL float4 *)xr)[2 * g];
                Q[i] = ((const LE_GLOBAL float4 *)xr)[2 * g + 1];
                if (a.up) {
                    const LE_GLOBAL float4 *ur = (const LE_GLOBAL float4 *)(a.up + src * K);
                    P[i] = le_silu_mul4(P[i], ur[2 * g]);
                    Q[i] = le_silu_mul4(Q[i], ur[2 * g + 1]);
                }
            } else {
                P[i] = Q[i] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
#pragma unroll
        for (int i = 0; i < XG; i++) am = fmaxf(am, amax8(P[i], Q[i]));
    } else if (live) {
        for (int i = tid; i < K / 4; i += 256) {
            float4 v = ((const LE_GLOBAL float4 *)xr)[i];
            if (a.up) v = le_silu_mul4(v, ((const LE_GLOBAL float4 *)(a.up + src * K))[i]);
            am = fmaxf(am, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) am = fmaxf(am, __shfl_xor(am, o));
    if (lane == 0) red[tid >> 6] = am;
    __syncthreads();
    am = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    int ex = 0;
    if (am > 0.f && am <= 3.0e38f) {
        (void)frexpf(am, &ex); /* am = f 2^ex, f in [0.5, 1) */
        ex = max(ex - 7, -100);
    }
    const float sc = live ? ldexpf(1.f, -ex) : 0.f;
    _Float16 *A = (_Float16 *)ws;
    u8 *S = ws + gq_s_off(a.mp, K);
    auto convert = [&](int g, float4 p, float4 q) { gq_xconvert<SK>(g, p, q, sc, t, K, A, S); };
    if (inreg) {
#pragma unroll
        for (int i = 0; i < XG; i++) {
            const int g = tid + 256 * i;
            if (g < ng) convert(g, P[i], Q[i]);
        }
    } else {
        for (int g = tid; g < ng; g += 256) {
            float4 p = make_float4(0.f, 0.f, 0.f, 0.f), q = p;
            if (live) {
                p = ((const LE_GLOBAL float4 *)xr)[2 * g];
                q = ((const LE_GLOBAL float4 *)xr)[2 * g + 1];
                if (a.up) {
                    const LE_GLOBAL float4 *ur = (const LE_GLOBAL float4 *)(a.up + src * K);
                    p = le_silu_mul4(p, ur[2 * g]);
                    q = le_silu_mul4(q, ur[2 * g + 1]);
                }
            }
            convert(g, p, q);
        }
    }
    if (tid == 0) {
        constexpr int srec = SK == 0 ? 0 : SK == 1 ? 1024 : 2048;
        ((float *)(ws + gq_t_off(a.mp, K, srec)))[t] = live ? ldexpf(1.f, ex) : 0.f;
    }
}

/* Grouped form, K <= 4096: one wave per pair (four per block), each lane holding up to 8 groups of
 * the pair's row; the largest magnitude by a wave reduction (no block barrier), then the same
 * conversion as gq_xprep_body, so the same bits. */
template <int SK>
__device__ __forceinline__ void gq_xprepw_body(const GqArgs &a, u8 *ws) {
    const int K = a.cols, lane = threadIdx.x & 63;
    const int p = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (p >= a.npair) return; /* wave-uniform; no block barrier below */
    const int srcp = a.in_idx[p]; /* loads with the slots' offsets */
    int o0, first;
    const int lo = le_slot_walk(a.off, a.nslot, a.bm, [p](int b, int e, int, int) { return p >= b && p < e; }, o0, first);
    if (lo < 0) return;
    const int j = p - o0, tile = first + j / a.bm;
    if (tile >= a.maxt) return;
    const int t = tile * a.bm + j % a.bm;
    const LE_GLOBAL float *xr = (const LE_GLOBAL float *)(a.x + (size_t)srcp * K);
    constexpr int XW = 8;
    const int ng = K / 8;
    float4 P[XW], Q[XW];
    float am = 0.f;
#pragma unroll
    for (int i = 0; i < XW; i++) {
        const int g = lane + 64 * i;
        if (g < ng) {
            P[i] = ((const LE_GLOBAL float4 *)xr)[2 * g];
            Q[i] = ((const LE_GLOBAL float4 *)xr)[2 * g + 1];
            if (a.up) {
                const LE_GLOBAL float4 *ur = (const LE_GLOBAL float4 *)(a.up + (size_t)srcp * K);
                P[i] = le_silu_mul4(P[i], ur[2 * g]);
                Q[i] = le_silu_mul4(Q[i], ur[2 * g + 1]);
            }
        } else {
            P[i] = Q[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        am = fmaxf(am, amax8(P[i], Q[i]));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) am = fmaxf(am, __shfl_xor(am, o));
    int ex = 0;
    if (am > 0.f && am <= 3.0e38f) {
        (void)frexpf(am, &ex); /* am = f 2^ex, f in [0.5, 1) */
        ex = max(ex - 7, -100);
    }
    const float sc = ldexpf(1.f, -ex);
    _Float16 *A = (_Float16 *)ws;
    u8 *S = ws + gq_s_off(a.mp, K);
#pragma unroll
    for (int i = 0; i < XW; i++) {
        const int g = lane + 64 * i;
        if (g < ng) gq_xconvert<SK>(g, P[i], Q[i], sc, t, K, A, S); /* ng % 32 == 0: a sum's lanes are all in or all out */
    }
    if (lane == 0) {
        constexpr int srec = SK == 0 ? 0 : SK == 1 ? 1024 : 2048;
        ((float *)(ws + gq_t_off(a.mp, K, srec)))[t] = ldexpf(1.f, ex);
    }
}

/* Direct-to-LDS loads (gfx950 global_load_lds_dwordx4): the load unit writes lane l's 16 bytes
 * at M0 + 16 l, so a wave's 64 chunks land as one contiguous 1 KB run with no registers held
 * while in flight. Issued from inline assembly so the compiler does not wait for them before
 * every LDS read; the kernel waits for them explicitly (the memory counter retires loads in
 * issue order). */
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void gq_lds_dma16(const u8 *g, u32 lds_addr) {
    asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds_addr) : "memory", "m0");
}
#pragma clang diagnostic pop
template <int N>
__device__ __forceinline__ void gq_vm_wait() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ u32 gq_lds_addr(const void *p) { return (u32)(size_t)(const __attribute__((address_space(3))) void *)p; }

/* End of a block's tile: acc times the token scales into y, the K slice's partial results or (neither)
 * atomically added into y. LDSB: bytes of LDS that may be overwritten. CUT: rows below rmin are left out (compared
 * for every block, the check cost the short slices of the other kernels 1-2 us: 4096 x 4096 M = 256 Q3_K 34.5 against
 * 33.0, Q8_0 39.0 / 37.9). */
template <int WM, int WN, int TM, int TN, bool GR, int LDSB, bool CUT = false>
__device__ __forceinline__ void gq_store(const GqArgs &a, u8 *lds, const float *tsc, const le_v16f (&acc)[TM][TN], int M, int mb,
                                         int nb, int pair0, bool second, int rmin = 0) {
    constexpr int BN = 32 * TN * WN, NT = 64 * WM * WN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave / WN, wn = wave % WN;
    const int n = lane & 31, hs = lane >> 5;
    /* D lane l element e: token 8 (e / 4) + 4 (l / 32) + e % 4 of the tile, row l % 32; the
     * token scales of the padded tile are all loaded first (one memory round trip) */
    float ts[TM][16];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int e = 0; e < 16; e++) ts[i][e] = tsc[mb + (wm * TM + i) * 32 + 4 * hs + 8 * (e >> 2) + (e & 3)];
    if (!GR && a.ksplit > 1 && !a.part) { /* K slices without a partial-result buffer: atomic adds */
#pragma unroll
        for (int i = 0; i < TM; i++) {
            const int t0 = mb + (wm * TM + i) * 32 + 4 * hs;
#pragma unroll
            for (int k = 0; k < TN; k++) {
                const int r = nb + (wn * TN + k) * 32 + n;
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const int t = t0 + 8 * (e >> 2) + (e & 3);
                    if (t < M && (!CUT || r >= rmin) && r < a.rows) unsafeAtomicAdd(a.y + (size_t)t * a.rows + r, acc[i][k][e] * ts[i][e]);
                }
            }
        }
        return;
    }
    /* Stores through LDS, one 32-token tile of every wave row at a time: the waves place their
     * results as [token][row] (row stride BN + 8 floats: the two 4-token halves of a fragment fall
     * on different banks), then each token's BN outputs leave as 16-byte stores of consecutive
     * rows (a wave covers 1 KB of one output row) instead of 4-byte stores 32 to a row. */
    float *dst = (!GR && a.ksplit > 1) ? a.part + (size_t)blockIdx.y * a.m * a.rows : second ? a.y2 : a.y;
    constexpr int TS = BN + 8, NQ = BN / 4;
    static_assert((size_t)WM * 32 * TS * 4 <= (size_t)LDSB, "output staging must fit the step buffers");
    float *T = (float *)lds;
    const bool vec = (a.rows & 3) == 0 && ((size_t)dst & 15) == 0;
#pragma unroll
    for (int i = 0; i < TM; i++) {
        __syncthreads(); /* the step buffers (or the previous round) are no longer read */
#pragma unroll
        for (int k = 0; k < TN; k++) {
            const int rl = (wn * TN + k) * 32 + n;
#pragma unroll
            for (int e = 0; e < 16; e++)
                T[(wm * 32 + 4 * hs + 8 * (e >> 2) + (e & 3)) * TS + rl] = acc[i][k][e] * ts[i][e];
        }
        __syncthreads();
        for (int c = tid; c < WM * 32 * NQ; c += NT) {
            const int tl = c / NQ, q = c - tl * NQ;
            const int t = mb + ((tl >> 5) * TM + i) * 32 + (tl & 31), r = nb + 4 * q;
            if (t >= M || r >= a.rows) continue;
            int o = t;
            if constexpr (GR) o = a.out_idx[pair0 + t - mb];
            const float4 v = *(const float4 *)(T + tl * TS + 4 * q);
            float *yp = dst + (size_t)o * a.rows + r;
            if (vec && (!CUT || r >= rmin) && r + 3 < a.rows) {
                *(float4 *)yp = v;
            } else {
                const float vv[4] = {v.x, v.y, v.z, v.w};
                for (int u = 0; u < 4 && r + u < a.rows; u++)
                    if (!CUT || r + u >= rmin) yp[u] = vv[u];
            }
        }
    }
}

/* ============================ main kernel ============================ */
/* NA > 0: the activation fragments go straight to LDS, a ring of NA step slots (2: loaded one
 * step ahead, issued as the step starts, in the LDS the register-staged form uses for them; 3:
 * two steps ahead, with the weights' loads) instead of through registers; the weights keep the
 * register staging. Every launched kernel uses NA = 2 (measured against registers at M=512: Q4_K
 * 109 -> 95 us, Q6_K 147 -> 114, Q8_0 252 -> 230, IQ2_XXS 98 -> 92; the three-slot ring 100 us for
 * Q4_K); the results are the same bits in every form. */
/* UA: only the tiles whose weights are not 16-byte aligned (gqu_body) */
template <int TY, int WM, int WN, int TM, int TN, bool GR = false, int NA = 0, bool UA = false>
__device__ __forceinline__ void gq_body(const GqArgs &a, const u8 *ws, const int id) {
    using F = GqF<TY>;
    constexpr bool AD = NA > 0;
    static_assert(NA == 0 || NA == 2 || NA == 3, "activation ring of 2 or 3 slots");
    constexpr int BM = 32 * TM * WM, BN = 32 * TN * WN, NT = 64 * WM * WN;
    constexpr int WB = BN * F::SLOT, AB = BM * 256, BUF = AD ? WB : WB + AB;
    constexpr int SBYTES = F::SREC ? (BM / 32) * F::SREC : 0; /* per super-block */
    constexpr int NWC = (BN * F::NCH + NT - 1) / NT, NAC = AB / 16 / NT, NSC = (SBYTES / 16 + NT - 1) / NT;
    static_assert(AB / 16 % NT == 0, "activation chunks must divide over the threads");
    extern __shared__ uint4 smem[];
    u8 *lds = (u8 *)smem;
    u8 *Aring = lds + 2 * BUF;          /* NA > 0: [NA][AB] activation step slots */
    u8 *Sl = lds + 2 * BUF + NA * AB;  /* [2][SBYTES] sum records, by super-block parity */
    u8 *tab = Sl + 2 * SBYTES;          /* IQ tables */

    const int K = a.cols, nsb = K >> 8;
    const int NTR1 = (a.rows + BN - 1) / BN, NTR = GR && a.dual ? 2 * NTR1 : NTR1, MT = GR ? a.maxt : (a.m + BM - 1) / BM;
    /* 8 or more row tiles: blocks of one row tile (its token tiles) share blockIdx % 8, the XCD
     * and its L2; fewer: row tiles vary fastest, so consecutive blocks spread over every XCD */
    const int j = id >> 3;
    const int mt = NTR >= 8 ? j % MT : id / NTR, nt = NTR >= 8 ? (j / MT) * 8 + (id & 7) : id % NTR;
    if (nt >= NTR || mt >= MT) return; /* uniform over the block */
    const bool second = nt >= NTR1; /* dual grouped form: a row tile of the second weight set */
    const int nb = (second ? nt - NTR1 : nt) * BN, mb = mt * BM;
    /* tokens of this tile: M = all tokens (plain), or the tile's pairs (grouped: rows of its slot) */
    int M = a.m, pair0 = 0;
    const u8 *Wsrc = a.w;
    if constexpr (GR) {
        int sl;
        if (!le_tile_of(a.off, a.nslot, a.bm, mt, sl, pair0)) return; /* uniform: past the last tile */
        M = mb + min(BM, a.off[sl + 1] - pair0); /* token t of the tile is valid while t < M */
        if (second)
            Wsrc = a.ptrs2 ? a.ptrs2[sl] : a.w2 + (size_t)sl * a.w_slot_bytes;
        else
            Wsrc = a.ptrs ? a.ptrs[sl] : a.w + (size_t)sl * a.w_slot_bytes;
        if (UA && ((size_t)Wsrc & 15) == 0) return;
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const size_t rb = (size_t)nsb * F::SBB;
    const int sb0 = blockIdx.y * (nsb / a.ksplit), sb1 = sb0 + nsb / a.ksplit;
    const int nstep = 2 * sb1;
    const u8 *Ag = ws;
    const u8 *Sg = ws + gq_s_off(a.mp, K);
    const float *tsc = (const float *)(ws + gq_t_off(a.mp, K, F::SREC));

    if constexpr (F::TAB > 0) gq_tables<TY>(tab);

    struct Set {
        uint4 w[NWC], x[AD ? 1 : NAC], s[NSC > 0 ? NSC : 1];
    };
    /* every load is unconditional (addresses clamped) so the waits before staging count exactly
     * the loads of the step being staged; steps past the slice re-read the last one. Even steps
     * (first halves of super-blocks, always set RB) also bring the super-block's sum records. */
    /* per-thread 32-bit load offsets, computed once (the host keeps a slice's weights and the
     * activation planes below 4 GiB): so each load is a scalar base plus one of these */
    u32 wo0[NWC], wo1[NWC], xo[NAC], so[NSC > 0 ? NSC : 1];
    bool xlive[NAC];
#pragma unroll
    for (int i = 0; i < NWC; i++) {
        const int c = min(tid + NT * i, BN * F::NCH - 1), row = c / F::NCH, k = c - row * F::NCH;
        const u32 base = (u32)min(nb + row, a.rows - 1) * (u32)rb;
        wo0[i] = base + F::goff(k, 0);
        wo1[i] = base + F::goff(k, 1);
    }
#pragma unroll
    for (int i = 0; i < NAC; i++) {
        const int c = tid + NT * i, tl = c >> 9, off = c & 511; /* 512 chunks = 8 KB per 32-token tile */
        xo[i] = (u32)(mb / 32 + tl) * (u32)(K / 16) * 1024u + 16u * off;
        xlive[i] = mb + 32 * tl + (off & 31) < M; /* fragment lane l holds token l % 32 */
    }
#pragma unroll
    for (int i = 0; i < (NSC > 0 ? NSC : 1); i++) {
        const int c = min(tid + NT * i, SBYTES > 0 ? SBYTES / 16 - 1 : 0), tl = c / (F::SREC > 0 ? F::SREC / 16 : 1);
        const int off = c - tl * (F::SREC > 0 ? F::SREC / 16 : 1);
        so[i] = (u32)(mb / 32 + tl) * (u32)nsb * (u32)F::SREC + 16u * off;
    }
    auto issue = [&](int s_, Set &R, bool even) {
        const int s = min(s_, nstep - 1), sb = s >> 1, h = s & 1;
        const u8 *w0 = Wsrc + (size_t)sb * F::SBB;
#pragma unroll
        for (int i = 0; i < NWC; i++) {
            const u8 *p = w0 + (h ? wo1[i] : wo0[i]);
            R.w[i] = F::ALIGNED ? ldg16c(p) : ldg16u(p); /* cached: the next step reads the same lines */
        }
        if constexpr (!AD) {
            const u8 *x0 = Ag + (size_t)(sb * 16 + 8 * h) * 1024;
#pragma unroll
            for (int i = 0; i < NAC; i++) R.x[i] = ldg16c(x0 + xo[i]);
        }
        if (SBYTES > 0 && even) {
            const u8 *s0p = Sg + (size_t)sb * F::SREC;
#pragma unroll
            for (int i = 0; i < NSC; i++) R.s[i] = ldg16c(s0p + so[i]);
        }
    };
    auto stage = [&](int s, const Set &R, bool even) {
        const int sb = s >> 1, h = s & 1;
        u8 *B = lds + h * BUF;
#pragma unroll
        for (int i = 0; i < NWC; i++) {
            const int c = tid + NT * i;
            if (NWC * NT > BN * F::NCH && c >= BN * F::NCH) break;
            const int row = c / F::NCH, k = c - row * F::NCH;
            *(uint4 *)(B + row * F::SLOT + F::loff(k)) = R.w[i];
        }
        if constexpr (!AD) {
#pragma unroll
            for (int i = 0; i < NAC; i++) ((uint4 *)(B + WB))[tid + NT * i] = R.x[i];
        }
        if constexpr (SBYTES > 0) {
            if (even) {
#pragma unroll
                for (int i = 0; i < NSC; i++) {
                    const int c = tid + NT * i;
                    if (NSC * NT > SBYTES / 16 && c >= SBYTES / 16) break;
                    ((uint4 *)(Sl + (sb & 1) * SBYTES))[c] = R.s[i];
                }
            }
        }
    };

    /* NA > 0: step s_'s activation fragments into ring slot s_ % NA (steps past the slice re-read
     * the last one into a slot that is no longer read) */
    auto dma = [&](int s_) {
        if constexpr (AD) {
            const int s = min(s_, nstep - 1), sb = s >> 1, h = s & 1;
            const u8 *x0 = Ag + (size_t)(sb * 16 + 8 * h) * 1024;
            u8 *dst = Aring + (s_ % (NA > 0 ? NA : 1)) * AB + 64 * 16 * wave;
#pragma unroll
            for (int i = 0; i < NAC; i++) { /* the LDS address is uniform over the wave (M0) */
                const u32 la = __builtin_amdgcn_readfirstlane(gq_lds_addr(dst + NT * 16 * i));
                /* lanes of tokens past the tile's last one load nothing: their LDS bytes only
                 * reach output rows that are never stored, and a 128-byte line holds 8 tokens,
                 * so a sparse tile (grouped form) fetches a quarter of the lines per valid 8 */
                if (xlive[i]) gq_lds_dma16(x0 + xo[i], la);
            }
        }
    };

    /* SEP: a super-block's products in an accumulator of their own, which joins acc at its end. A wave of one 32 x 32
     * tile has the registers for it; a shared one lay in accumulation registers there, so that each rescaling moved it
     * out and back, before the wave's one chain of MFMAs went on (24 tokens, 2560 x 6912, against this form: Q3_K 53.5 /
     * 48.9 us, Q5_K 56.5 / 51.5, IQ3_XXS 65.3 / 61.0; 14336 x 4096 Q3_K 26.6 / 25.5). */
    constexpr bool SEP = F::EPI == 1 && TM * TN == 1;
    le_v16f acc[TM][TN], d1[SEP ? TM : 1][SEP ? TN : 1];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int k = 0; k < TN; k++) acc[i][k] = (le_v16f){};

    const int n = lane & 31, hs = lane >> 5;
    int rowS[TN]; /* Q8_0 / Q4_0: the accumulator holds the row's sum times 2^rowS */
#pragma unroll
    for (int k = 0; k < TN; k++) rowS[k] = 127;
    /* EPI == 1: the accumulator holds the row's sum in units of unit[k], the super-block scale in use;
     * live[k]: all ones, or zero while the super-block's scale is zero (its codes then count as zero) */
    float unit[TN];
    u32 live[TN];
#pragma unroll
    for (int k = 0; k < TN; k++) unit[k] = 1.f, live[k] = SEP ? ~0u : 0;
    Set RA, RB; /* RA holds odd (h = 1) steps, RB even ones */
    const int s0 = 2 * sb0;
    /* the loads must reach the memory pipeline in step order (RA's before RB's, as in the loop),
     * or the wait at the loop head would have to cover both sets: no reordering across issues */
    issue(s0, RB, true);
    dma(s0);
    stage(s0, RB, true);
    issue(s0 + 1, RA, false);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (NA == 3) dma(s0 + 1);
    issue(s0 + 2, RB, true);
    __builtin_amdgcn_sched_barrier(0);

    for (int sb = sb0; sb < sb1; sb++) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int s = 2 * sb + h;
            /* this step's activations: younger are the loads of steps s + 2 (weights) and, with
             * three slots, s + 1 (activations) */
            if constexpr (NA == 3) {
                if (h == 0) gq_vm_wait<NWC + NAC + (SBYTES > 0 ? NSC : 0)>();
                else gq_vm_wait<NWC + NAC>();
            } else if constexpr (NA == 2) {
                if (h == 0) gq_vm_wait<NWC + (SBYTES > 0 ? NSC : 0)>();
                else gq_vm_wait<NWC>();
            }
            gq_barrier(); /* step s is staged; every wave is done with step s-1's buffer */
            if constexpr (NA == 2) dma(s + 1); /* slot (s + 1) % 2 was last read in step s - 1 */
            const u8 *Wb = lds + h * BUF, *Ab = (AD ? Aring + (s % (NA > 0 ? NA : 1)) * AB : Wb + WB) + (wm * TM) * 8192;
            const u8 *rs[TN];
#pragma unroll
            for (int k = 0; k < TN; k++) rs[k] = Wb + (wn * TN * 32 + 32 * k + n) * F::SLOT;
            /* The step's eight chunks in the order the decoders produce them (Q4_K, Q5_K: low and high
             * nibbles of the same bytes, chunks c and c + 2, together). The activation fragments of the
             * next chunk are read while this chunk's MFMAs run (read right before their use, each MFMA
             * waited out an LDS read). */
            le_v8h Af[2][TM];
            auto aread = [&](int p, le_v8h (&A)[TM]) {
                constexpr bool PAIR = TY == LE_TYPE_Q4_K || TY == LE_TYPE_Q5_K;
                const int c = TY == LE_TYPE_Q6_K ? 2 * (p & 3) + (p >> 2) : PAIR ? (p & 4) | ((p & 1) << 1) | ((p >> 1) & 1) : p;
#pragma unroll
                for (int i = 0; i < TM; i++) A[i] = as_v8h(*(const uint4 *)(Ab + i * 8192 + c * 1024 + lane * 16));
            };
            auto mma = [&](int p, const le_v8h (&B)[TN]) { /* position p of that order */
                if constexpr (SEP) { /* one MFMA a fragment: nothing to read behind */
                    le_v8h A[TM];
                    aread(p, A);
                    gq_mma(d1, A, B, h == 0 && p == 0);
                } else {
                    if (p < 7) aread(p + 1, Af[(p + 1) & 1]);
                    __builtin_amdgcn_sched_barrier(0x016); /* LDS reads stay on their side of the MFMAs; VALU, SALU and VMEM may cross */
                    gq_mma(acc, Af[p & 1], B, false);
                    __builtin_amdgcn_sched_barrier(0x016);
                }
            };
            if constexpr (!SEP) aread(0, Af[0]);
            /* stage the next step and issue the loads two steps ahead once this step's first
             * fragments are under way */
            auto pipe = [&]() {
                /* unconditional (a branch here would make the compiler wait for every load in
                 * flight): past the slice's end this stages a re-read into the buffer that is
                 * no longer read */
                if (h) stage(s + 1, RB, true);
                else stage(s + 1, RA, false);
                __builtin_amdgcn_sched_barrier(0);
                if (h) issue(s + 3, RB, true);
                else issue(s + 3, RA, false);
                if constexpr (NA == 3) dma(s + 2); /* slot (s + 2) % 3 was last read in step s - 1 */
                __builtin_amdgcn_sched_barrier(0);
            };
            if (F::EPI == 1 && !SEP && h == 0) {
                /* a new super-block scale: one multiplication puts the running sum into its units, so the
                 * MFMAs accumulate into it directly and a wave needs one accumulator, not a second one
                 * per super-block */
#pragma unroll
                for (int k = 0; k < TN; k++) {
                    const float d = F::scale(rs[k]);
                    live[k] = d == 0.f ? 0u : ~0u;
                    const float r = d == 0.f ? 1.f : unit[k] * __builtin_amdgcn_rcpf(d);
                    unit[k] = d == 0.f ? unit[k] : d;
#pragma unroll
                    for (int i = 0; i < TM; i++)
#pragma unroll
                        for (int e = 0; e < 16; e++) acc[i][k][e] *= r;
                }
            }
            if constexpr (TY == LE_TYPE_Q4_K) {
                const u32 mlo = 0x000F000Fu, mhi = 0x00F000F0u, c1024 = 0x64006400u;
                uint4 hd[TN];
                u32 scw[TN];
#pragma unroll
                for (int k = 0; k < TN; k++) {
                    hd[k] = *(const uint4 *)rs[k];
                    scw[k] = (h ? ((hd[k].w & 0x0F0F0F0Fu) | ((hd[k].y >> 2) & 0x30303030u)) : (hd[k].y & 0x3F3F3F3Fu)) & live[k];
                }
#pragma unroll
                for (int g = 0; g < 2; g++) {
                    uint4 kc[TN]; /* (sc_lo, -1024 sc_lo, sc_hi / 16, -64 sc_hi) as duplicated halves */
#pragma unroll
                    for (int k = 0; k < TN; k++) {
                        const u32 slo = pk_add(h1024_dup(scw[k], 2 * g), 0xE400E400u);
                        const u32 shi = pk_add(h1024_dup(scw[k], 2 * g + 1), 0xE400E400u);
                        kc[k] = make_uint4(slo, pk_mul(slo, 0xE400E400u), pk_mul(shi, 0x2C002C00u), pk_mul(shi, 0xD400D400u));
                    }
#pragma unroll
                    for (int c1 = 0; c1 < 2; c1++) {
                        le_v8h blo[TN], bhi[TN];
#pragma unroll
                        for (int k = 0; k < TN; k++) {
                            const uint2 q = *(const uint2 *)(rs[k] + 16 + 32 * g + 16 * c1 + 8 * hs);
                            const u32 ws_[2] = {q.x, q.y};
                            u32 l[4], hh[4];
#pragma unroll
                            for (int e = 0; e < 2; e++) {
                                const u32 x = ws_[e], x8 = x >> 8;
                                l[2 * e] = pk_fma(and_or(x, mlo, c1024), kc[k].x, kc[k].y);
                                l[2 * e + 1] = pk_fma(and_or(x8, mlo, c1024), kc[k].x, kc[k].y);
                                hh[2 * e] = pk_fma(and_or(x, mhi, c1024), kc[k].z, kc[k].w);
                                hh[2 * e + 1] = pk_fma(and_or(x8, mhi, c1024), kc[k].z, kc[k].w);
                            }
                            blo[k] = as_v8h(make_uint4(l[0], l[1], l[2], l[3]));
                            bhi[k] = as_v8h(make_uint4(hh[0], hh[1], hh[2], hh[3]));
                        }
                        mma(4 * g + 2 * c1, blo);
                        mma(4 * g + 2 * c1 + 1, bhi);
                        if (g == 0 && c1 == 0) pipe();
                    }
                }
            } else if constexpr (TY == LE_TYPE_Q6_K) {
                /* chunk c of half h uses sc[8h + c], as sc / 64 duplicated (exact) */
                u32 sp[TN][8];
#pragma unroll
                for (int k = 0; k < TN; k++) {
                    const uint2 sv = *(const uint2 *)(rs[k] + 96 + 8 * h);
                    const u32 sw[2] = {(sv.x & live[k]) ^ 0x80808080u, (sv.y & live[k]) ^ 0x80808080u};
#pragma unroll
                    for (int c = 0; c < 8; c++)
                        sp[k][c] = pk_mul(pk_add(h1024_dup(sw[c >> 2], c & 3), 0xE480E480u), 0x24002400u); /* (byte - 1152) / 64 */
                }
#pragma unroll
                for (int c1 = 0; c1 < 2; c1++) {
                    const int l0 = 16 * c1 + 8 * hs;
                    uint2 qa[TN], qb[TN], qh[TN];
#pragma unroll
                    for (int k = 0; k < TN; k++) {
                        qa[k] = *(const uint2 *)(rs[k] + l0);
                        qb[k] = *(const uint2 *)(rs[k] + 32 + l0);
                        qh[k] = *(const uint2 *)(rs[k] + 64 + l0);
                    }
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const int c = 2 * q + c1;
                        le_v8h B[TN];
#pragma unroll
                        for (int k = 0; k < TN; k++) {
                            const uint2 src = q & 1 ? qb[k] : qa[k];
                            const u32 sx = src.x >> (4 * (q >> 1)), sy = src.y >> (4 * (q >> 1));
                            const u32 hx = q < 2 ? (qh[k].x << (4 - 2 * q)) : (qh[k].x >> (2 * q - 4));
                            const u32 hy = q < 2 ? (qh[k].y << (4 - 2 * q)) : (qh[k].y >> (2 * q - 4));
                            const u32 vx = and_or(sx, 0x0F0F0F0Fu, hx & 0x30303030u);
                            const u32 vy = and_or(sy, 0x0F0F0F0Fu, hy & 0x30303030u);
                            /* (1024 + q6) - 1056 = q6 - 32 exactly, then one rounding by sc / 64 */
                            const u32 sc = sp[k][c];
                            B[k] = as_v8h(make_uint4(pk_mul(pk_add(h1024_02(vx), 0xE420E420u), sc), pk_mul(pk_add(h1024_13(vx), 0xE420E420u), sc),
                                                     pk_mul(pk_add(h1024_02(vy), 0xE420E420u), sc), pk_mul(pk_add(h1024_13(vy), 0xE420E420u), sc)));
                        }
                        mma(4 * c1 + q, B);
                        if (c1 == 0 && q == 0) pipe();
                    }
                }
            } else if constexpr (TY == LE_TYPE_Q8_0 || TY == LE_TYPE_Q4_0) {
                /* per-32 scales inside the codes: fp16(q * d_b 2^S) (one rounding), with a power of two
                 * 2^S per row that keeps every code inside the fp16 range whatever the scales are:
                 * S only decreases, to the value that puts the step's largest |d_b| 2^S in
                 * [128, 256) (|q| <= 128) when that is below the current one, and the accumulator
                 * is then rescaled (a wave-uniform branch, taken at the first step and
                 * otherwise only when a row's scales grow); the result is multiplied by 2^-S */
                constexpr int DO = TY == LE_TYPE_Q8_0 ? 128 : 64, QB = TY == LE_TYPE_Q8_0 ? 32 : 16;
                u32 r[TN][4];
                bool grow = false;
                int sn[TN];
#pragma unroll
                for (int k = 0; k < TN; k++) {
                    u32 dv[4], mx = 0;
#pragma unroll
                    for (int b = 0; b < 4; b++) {
                        dv[b] = *(const u32 *)(rs[k] + DO + 16 * b) & 0xFFFFu;
                        mx = max(mx, dv[b] & 0x7FFFu);
                    }
                    const int e = max((int)(mx >> 10), 1); /* biased fp16 exponent of the largest |d_b| */
                    sn[k] = min(rowS[k], 22 - e);
                    grow |= sn[k] != rowS[k];
                    const float up_ = __builtin_bit_cast(float, (u32)(127 + sn[k]) << 23);
#pragma unroll
                    for (int b = 0; b < 4; b++) r[k][b] = h2dup(h2f(dv[b]) * up_);
                }
                if (__any(grow)) {
#pragma unroll
                    for (int k = 0; k < TN; k++) {
                        const float f = ldexpf(1.f, sn[k] - rowS[k]);
                        rowS[k] = sn[k];
#pragma unroll
                        for (int i = 0; i < TM; i++)
#pragma unroll
                            for (int e = 0; e < 16; e++) acc[i][k][e] *= f;
                    }
                }
#pragma unroll
                for (int b = 0; b < 4; b++) {
#pragma unroll
                    for (int c1 = 0; c1 < 2; c1++) {
                        const int c = 2 * b + c1;
                        le_v8h B[TN];
#pragma unroll
                        for (int k = 0; k < TN; k++) {
                            if constexpr (TY == LE_TYPE_Q8_0) {
                                const uint2 q = *(const uint2 *)(rs[k] + QB * b + 16 * c1 + 8 * hs);
                                const u32 x = q.x ^ 0x80808080u, y = q.y ^ 0x80808080u; /* q + 128 */
                                B[k] = as_v8h(make_uint4(pk_mul(pk_add(h1024_02(x), 0xE480E480u), r[k][b]), pk_mul(pk_add(h1024_13(x), 0xE480E480u), r[k][b]),
                                                         pk_mul(pk_add(h1024_02(y), 0xE480E480u), r[k][b]), pk_mul(pk_add(h1024_13(y), 0xE480E480u), r[k][b])));
                            } else { /* value j < 16: low nibble of byte j; j >= 16: high nibble of byte j - 16 */
                                const uint2 q = *(const uint2 *)(rs[k] + QB * b + 8 * hs);
                                const u32 x = (q.x >> (4 * c1)) & 0x0F0F0F0Fu, y = (q.y >> (4 * c1)) & 0x0F0F0F0Fu;
                                B[k] = as_v8h(make_uint4(pk_mul(pk_add(h1024_02(x), 0xE408E408u), r[k][b]), pk_mul(pk_add(h1024_13(x), 0xE408E408u), r[k][b]),
                                                         pk_mul(pk_add(h1024_02(y), 0xE408E408u), r[k][b]), pk_mul(pk_add(h1024_13(y), 0xE408E408u), r[k][b])));
                            }
                        }
                        mma(c, B);
                        if (c == 0) pipe();
                    }
                }
            } else if constexpr (TY == LE_TYPE_Q5_K) {
                /* the Q4_K decode with the fifth bit of each code from qh: bit 2G (low nibbles of group
                 * G) and 2G + 1 (high nibbles) of byte l (src/quant.rs:83-95); codes sc * q <= 1953 */
                u32 scw[TN];
#pragma unroll
                for (int k = 0; k < TN; k++) {
                    const uint4 hd = *(const uint4 *)rs[k];
                    scw[k] = (h ? ((hd.w & 0x0F0F0F0Fu) | ((hd.y >> 2) & 0x30303030u)) : (hd.y & 0x3F3F3F3Fu)) & live[k];
                }
#pragma unroll
                for (int g = 0; g < 2; g++) {
                    const int G = 2 * h + g;
                    uint4 kc[TN]; /* (sc_lo, -1024 sc_lo, sc_hi, -1024 sc_hi) as duplicated halves */
#pragma unroll
                    for (int k = 0; k < TN; k++) {
                        const u32 slo = pk_add(h1024_dup(scw[k], 2 * g), 0xE400E400u);
                        const u32 shi = pk_add(h1024_dup(scw[k], 2 * g + 1), 0xE400E400u);
                        kc[k] = make_uint4(slo, pk_mul(slo, 0xE400E400u), shi, pk_mul(shi, 0xE400E400u));
                    }
#pragma unroll
                    for (int c1 = 0; c1 < 2; c1++) {
                        le_v8h blo[TN], bhi[TN];
#pragma unroll
                        for (int k = 0; k < TN; k++) {
                            const uint2 q = *(const uint2 *)(rs[k] + 48 + 32 * g + 16 * c1 + 8 * hs);
                            const uint2 qh = *(const uint2 *)(rs[k] + 16 + 16 * c1 + 8 * hs);
                            const u32 lx = and_or(q.x, 0x0F0F0F0Fu, ((qh.x >> (2 * G)) << 4) & 0x10101010u);
                            const u32 ly = and_or(q.y, 0x0F0F0F0Fu, ((qh.y >> (2 * G)) << 4) & 0x10101010u);
                            const u32 hx = and_or(q.x >> 4, 0x0F0F0F0Fu, ((qh.x >> (2 * G + 1)) << 4) & 0x10101010u);
                            const u32 hy = and_or(q.y >> 4, 0x0F0F0F0Fu, ((qh.y >> (2 * G + 1)) << 4) & 0x10101010u);
                            blo[k] = as_v8h(make_uint4(pk_fma(h1024_02(lx), kc[k].x, kc[k].y), pk_fma(h1024_13(lx), kc[k].x, kc[k].y),
                                                       pk_fma(h1024_02(ly), kc[k].x, kc[k].y), pk_fma(h1024_13(ly), kc[k].x, kc[k].y)));
                            bhi[k] = as_v8h(make_uint4(pk_fma(h1024_02(hx), kc[k].z, kc[k].w), pk_fma(h1024_13(hx), kc[k].z, kc[k].w),
                                                       pk_fma(h1024_02(hy), kc[k].z, kc[k].w), pk_fma(h1024_13(hy), kc[k].z, kc[k].w)));
                        }
                        mma(4 * g + 2 * c1, blo);
                        mma(4 * g + 2 * c1 + 1, bhi);
                        if (g == 0 && c1 == 0) pipe();
                    }
                }
            } else if constexpr (TY == LE_TYPE_Q3_K) {
                /* value 128h + 32s + l: code ((qs[32h + l] >> 2s) & 3) - (hm[l] bit 4h + s ? 0 : 4), scale
                 * 8h + c of the sixteen signed 6-bit scales (src/quant.rs:113-126); |code * scale| <= 128, exact */
                u32 sp[TN][8];
#pragma unroll
                for (int k = 0; k < TN; k++) {
                    const uint4 sw = *(const uint4 *)(rs[k] + 64); /* scale byte i at slot byte 66 + i */
                    const u32 s0 = __builtin_amdgcn_alignbyte(sw.y, sw.x, 2), s1 = __builtin_amdgcn_alignbyte(sw.z, sw.y, 2);
                    const u32 s2 = __builtin_amdgcn_alignbyte(sw.w, sw.z, 2);
                    /* scale i = 8h + c: low 4 bits from byte c (h = 0) or its high nibble (h = 1), bits 4-5
                     * from byte 8 + c % 4 at bit 2 (2h + c / 4) */
                    const u32 v0 = ((s0 >> (4 * h)) & 0x0F0F0F0Fu) | (((s2 >> (4 * h)) & 0x03030303u) << 4);
                    const u32 v1 = ((s1 >> (4 * h)) & 0x0F0F0F0Fu) | (((s2 >> (4 * h + 2)) & 0x03030303u) << 4);
#pragma unroll
                    for (int c = 0; c < 8; c++) sp[k][c] = pk_add(h1024_dup(c < 4 ? v0 : v1, c & 3), 0xE420E420u) & live[k]; /* byte - 32 */
                }
                uint2 qa[TN][2], hm[TN][2];
#pragma unroll
                for (int k = 0; k < TN; k++)
#pragma unroll
                    for (int p = 0; p < 2; p++) {
                        qa[k][p] = *(const uint2 *)(rs[k] + 16 * p + 8 * hs);
                        hm[k][p] = *(const uint2 *)(rs[k] + 32 + 16 * p + 8 * hs);
                    }
#pragma unroll
                for (int c = 0; c < 8; c++) {
                    const int sub = c >> 1, p = c & 1;
                    le_v8h B[TN];
#pragma unroll
                    for (int k = 0; k < TN; k++) {
                        const u32 vx = and_or(qa[k][p].x >> (2 * sub), 0x03030303u, ((hm[k][p].x >> (4 * h + sub)) & 0x01010101u) << 2);
                        const u32 vy = and_or(qa[k][p].y >> (2 * sub), 0x03030303u, ((hm[k][p].y >> (4 * h + sub)) & 0x01010101u) << 2);
                        const u32 sc = sp[k][c];
                        B[k] = as_v8h(make_uint4(pk_mul(pk_add(h1024_02(vx), 0xE404E404u), sc), pk_mul(pk_add(h1024_13(vx), 0xE404E404u), sc),
                                                 pk_mul(pk_add(h1024_02(vy), 0xE404E404u), sc), pk_mul(pk_add(h1024_13(vy), 0xE404E404u), sc)));
                    }
                    mma(c, B);
                    if (c == 0) pipe();
                }
            } else if constexpr (TY == LE_TYPE_IQ2_S) {
                /* block 4h + b, 8-value group l: grid index qs[4b + l] | bits 2l, 2l+1 of qh[b] as bits 8-9,
                 * signs = byte 4b + l, factor 2 s + 1 of the block's nibble l / 2 (src/quant.rs:155-167) */
                const u8 *sgt = tab + 1024 * 16;
                u32 qhw[TN], scw[TN];
#pragma unroll
                for (int k = 0; k < TN; k++) {
                    qhw[k] = *(const u32 *)(rs[k] + 32 + 4 * h);
                    scw[k] = *(const u32 *)(rs[k] + 40 + 4 * h);
                }
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    u32 qi[TN], sg[TN];
#pragma unroll
                    for (int k = 0; k < TN; k++) {
                        qi[k] = *(const u32 *)(rs[k] + 4 * b);
                        sg[k] = *(const u32 *)(rs[k] + 16 + 4 * b);
                    }
#pragma unroll
                    for (int c1 = 0; c1 < 2; c1++) {
                        const int c = 2 * b + c1, l = 2 * c1 + hs;
                        le_v8h B[TN];
#pragma unroll
                        for (int k = 0; k < TN; k++) {
                            const u32 qhb = (qhw[k] >> (8 * b)) & 0xFFu;
                            const u32 gi = ((qi[k] >> (8 * l)) & 255u) | ((qhb << (8 - 2 * l)) & 0x300u);
                            const u32 f = pk_add(h1024_dup(2u * ((scw[k] >> (8 * b + 4 * c1)) & 15u) + 1u, 0), 0xE400E400u) & live[k];
                            const uint4 g = *(const uint4 *)(tab + 16 * gi);
                            const uint4 m = *(const uint4 *)(sgt + 16 * ((sg[k] >> (8 * l)) & 255u));
                            B[k] = as_v8h(make_uint4(pk_mul(g.x, f) ^ m.x, pk_mul(g.y, f) ^ m.y, pk_mul(g.z, f) ^ m.z, pk_mul(g.w, f) ^ m.w));
                        }
                        mma(c, B);
                        if (c == 0) pipe();
                    }
                }
            } else if constexpr (TY == LE_TYPE_IQ2_XXS || TY == LE_TYPE_IQ3_XXS) {
                constexpr int GB = TY == LE_TYPE_IQ2_XXS ? 16 : 8;
                const u8 *sgt = tab + 256 * GB;
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    uint2 rec[TN];
                    u32 aux[TN], f[TN];
#pragma unroll
                    for (int k = 0; k < TN; k++) {
                        if constexpr (TY == LE_TYPE_IQ2_XXS) {
                            rec[k] = *(const uint2 *)(rs[k] + 8 * b);
                            aux[k] = rec[k].y;
                        } else {
                            rec[k] = *(const uint2 *)(rs[k] + 8 * b);
                            aux[k] = *(const u32 *)(rs[k] + 32 + 4 * b);
                        }
                        f[k] = pk_add(h1024_dup(2u * (aux[k] >> 28) + 1u, 0), 0xE400E400u) & live[k]; /* (2s+1) */
                    }
#pragma unroll
                    for (int c1 = 0; c1 < 2; c1++) {
                        const int c = 2 * b + c1, l = 2 * c1 + hs;
                        le_v8h B[TN];
#pragma unroll
                        for (int k = 0; k < TN; k++) {
                            const uint4 m = *(const uint4 *)(sgt + 16 * ((aux[k] >> (7 * l)) & 127u));
                            uint4 g;
                            if constexpr (TY == LE_TYPE_IQ2_XXS) {
                                g = *(const uint4 *)(tab + GB * ((rec[k].x >> (8 * l)) & 255u));
                            } else {
                                const u32 iw = l < 2 ? rec[k].x : rec[k].y, sh = 16 * (l & 1);
                                const uint2 g0 = *(const uint2 *)(tab + GB * ((iw >> sh) & 255u));
                                const uint2 g1 = *(const uint2 *)(tab + GB * ((iw >> (sh + 8)) & 255u));
                                g = make_uint4(g0.x, g0.y, g1.x, g1.y);
                            }
                            B[k] = as_v8h(make_uint4(pk_mul(g.x, f[k]) ^ m.x, pk_mul(g.y, f[k]) ^ m.y, pk_mul(g.z, f[k]) ^ m.z,
                                                     pk_mul(g.w, f[k]) ^ m.w));
                        }
                        mma(c, B);
                        if (c == 0) pipe();
                    }
                }
            }
        }
        /* offset term of the super-block (the h = 1 buffer holds its second half and the header) */
        if constexpr (TY == LE_TYPE_Q4_K || TY == LE_TYPE_Q5_K) {
            const u8 *Wb = lds + BUF;
            const u8 *Sb = Sl + (sb & 1) * SBYTES + (wm * TM) * F::SREC;
#pragma unroll
            for (int k = 0; k < TN; k++) {
                const uint4 hd = *(const uint4 *)(Wb + (wn * TN * 32 + 32 * k + n) * F::SLOT);
                const u32 m0 = hd.z & 0x3F3F3F3Fu, m1 = ((hd.w >> 4) & 0x0F0F0F0Fu) | ((hd.z >> 2) & 0x30303030u);
                const le_v8h b2 = as_v8h(make_uint4(pk_add(h1024_02(m0), 0xE400E400u), pk_add(h1024_13(m0), 0xE400E400u),
                                                    pk_add(h1024_02(m1), 0xE400E400u), pk_add(h1024_13(m1), 0xE400E400u)));
                const float dm = SEP ? -h2f(hd.x >> 16) : -h2f(hd.x >> 16) * __builtin_amdgcn_rcpf(unit[k]);
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    const le_v8h a2 = as_v8h(*(const uint4 *)(Sb + i * 1024 + lane * 16));
                    const le_v16f d2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a2, b2, (le_v16f){}, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 16; e++) acc[i][k][e] = __builtin_fmaf(dm, d2[e], acc[i][k][e]);
                }
            }
        }
        if constexpr (SEP) {
            const float d = F::scale(lds + BUF + (wn * 32 + n) * F::SLOT);
#pragma unroll
            for (int e = 0; e < 16; e++) acc[0][0][e] = __builtin_fmaf(d, d1[0][0][e], acc[0][0][e]);
        }
    }
    if constexpr (AD) gq_vm_wait<0>(); /* no activation load may still be writing LDS */
    if constexpr (!SEP) {
#pragma unroll
        for (int k = 0; k < TN; k++) {
            const float f = F::EPI == 2 ? ldexpf(1.f, -rowS[k]) : unit[k];
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[i][k][e] *= f;
        }
    }
    gq_store<WM, WN, TM, TN, GR, 2 * BUF + NA * AB>(a, lds, tsc, acc, M, mb, nb, pair0, second);
}

/* Grouped form over a pointer table, behind the pipelined kernel: the tiles of the slots whose weights are not 16-byte
 * aligned, which loads straight to LDS do not take (the grouped launch's `ids` blocks dealt to this one's). The host
 * cannot look at a device table's entries; where all are aligned, as the tensors of a model file are, the blocks end
 * after one look at it (2 us a launch; handled inside the pipelined kernel, a second way to load cost its 128-pair
 * tiles 5-10% in spilled registers, and the check alone 2-3%: le_gpgt_*, with it, beside le_gpg_*). */
template <int TY, int WM, int WN, int TM, int TN>
__device__ __forceinline__ void gqu_body(const GqArgs &a, const u8 *ws) {
    const int lane = threadIdx.x & 63;
    u32 low = 0;
    for (int s = lane; s < a.nslot; s += 64) low |= (u32)(size_t)a.ptrs[s] | (a.ptrs2 ? (u32)(size_t)a.ptrs2[s] : 0u);
    if (!__any((int)(low & 15u))) return; /* uniform over the block: every wave looks at the whole table */
    for (int id = blockIdx.x; id < a.ids; id += gridDim.x) {
        gq_body<TY, WM, WN, TM, TN, true, 2, true>(a, ws, id);
        __syncthreads(); /* the tile's staging is no longer read */
    }
}

/* ============================ pipelined kernel ============================ */
/* Q4_K and Q5_K from 33 tokens: a block of 4 waves computes 32 TM tokens x 256 rows, each wave all the
 * tokens of 64 rows of its own (TN = 2).
 *
 * Why this shape. gq_body's 128 x 256 block has 8 waves of 128 x 32: every wave reads the whole
 * activation tile from LDS, 32 KB per 16-value chunk and CU, which takes as long as the chunk's MFMAs
 * (256 cycles at 128 B/cycle), and its fragment reads, decoding and MFMAs follow each other inside a
 * step that begins and ends at a barrier. Here a wave uses each activation fragment for two row
 * fragments (half the LDS reads), no row is decoded twice, and the stages of a 16-value position run one
 * position apart, so that LDS reads and decoding of later positions lie between the MFMAs of this one,
 * also across steps (128 values) and super-blocks.
 *
 * Position q of a step (8 positions of 16 values, in the decoder's order): weight bytes are read from
 * LDS two positions ahead, activation fragments and B fragments are ready one ahead. All global loads go
 * straight to LDS, a few per position (13 at once held up the wave's instructions). Activations: two step slots; the only barrier of a step sits between its
 * positions 6 and 7, when every wave has read its last activation fragment of the step and its loads of
 * the next one have landed. Weights: private to the wave, three step slots, loaded two steps ahead (a
 * register-staged form one step ahead was bound by their latency: 88 against 79 us at M = 512; the 2-byte
 * aligned formats cannot be loaded straight to LDS and stay on gq_body, where they measured 1-15%
 * faster than here). The accumulator holds a row's sum in units of the super-block scale; the offset
 * term of one tile per position is added beside the MFMAs.
 *
 * Measured, whole calls (pre-pass and slice sums included) on weights that no cache holds, in turn with gq_body's best
 * tile, 14336 x 4096: Q4_K M = 64 30.6 -> 29.1 us, 128 41.9 -> 38.3, 256 62.8 -> 54.2, 512 92.9 -> 78.9 (762 TFLOP/s); Q5_K
 * M = 512 98.3 -> 82.5. Under a benchmark's minutes of load, where the clock falls, 4% of M = 512 are left (96.8 ->
 * 93.0). Counters of the launch at M = 512 (profiles/counters_gemm_few_tokens.md): matrix cores busy 38% of the SIMD
 * cycles (gq_body 33%), half its LDS instructions, 0.8 conflict cycles each; its 448 blocks are a round and three
 * quarters of the 256 CUs. */
/* bytes of a staged row per step (its header in front: 16-byte pieces of half super-block 0; of half 1
 * the same 64 bytes further, where the header's place holds bytes that are not used) */
template <int TY>
constexpr int gp_slot() { return TY == LE_TYPE_Q4_K ? 80 : 112; }

/* Decoder state of one 32-row fragment (lane: row rs, K half hs). head: LDS reads of a super-block's
 * header; prep: take it (h = 0) or its second half's scales (h = 1) into use; fetch(q): LDS reads for
 * position q; frag(q): its B fragment. */
template <int TY>
struct GpD;

template <>
struct GpD<LE_TYPE_Q4_K> {
    uint4 nh;
    u32 scw, sc1, live;
    le_v8h b2;   /* mins of the super-block as exact halves */
    float d, dm; /* its scale, and -offset scale (prep of the kernel: over the unit in use) */
    uint2 raw[2];
    uint4 kc;
    __device__ __forceinline__ void head(const u8 *rs, int) { nh = *(const uint4 *)rs; }
    __device__ __forceinline__ void prep(int h) {
        if (h == 0) {
            d = h2f(nh.x & 0xFFFFu);
            live = d == 0.f ? 0u : ~0u;
            scw = nh.y & 0x3F3F3F3Fu & live;
            sc1 = ((nh.w & 0x0F0F0F0Fu) | ((nh.y >> 2) & 0x30303030u)) & live;
            const u32 m0 = nh.z & 0x3F3F3F3Fu, m1 = ((nh.w >> 4) & 0x0F0F0F0Fu) | ((nh.z >> 2) & 0x30303030u);
            b2 = as_v8h(make_uint4(pk_add(h1024_02(m0), 0xE400E400u), pk_add(h1024_13(m0), 0xE400E400u),
                                   pk_add(h1024_02(m1), 0xE400E400u), pk_add(h1024_13(m1), 0xE400E400u)));
            dm = -h2f(nh.x >> 16);
        } else {
            scw = sc1;
        }
    }
    __device__ __forceinline__ void fetch(const u8 *rs, int q, int hs) {
        if ((q & 1) == 0) raw[(q >> 1) & 1] = *(const uint2 *)(rs + 16 + 32 * (q >> 2) + 16 * ((q >> 1) & 1) + 8 * hs);
    }
    __device__ __forceinline__ le_v8h frag(int q, int, u32 mlo, u32 mhi, u32 c) {
        if ((q & 3) == 0) { /* (sc_lo, -1024 sc_lo, sc_hi / 16, -64 sc_hi) as duplicated halves */
            const int g = q >> 2;
            const u32 slo = pk_add(h1024_dup(scw, 2 * g), 0xE400E400u), shi = pk_add(h1024_dup(scw, 2 * g + 1), 0xE400E400u);
            kc = make_uint4(slo, pk_mul(slo, 0xE400E400u), pk_mul(shi, 0x2C002C00u), pk_mul(shi, 0xD400D400u));
        }
        const uint2 r = raw[(q >> 1) & 1];
        const u32 m = q & 1 ? mhi : mlo, f = q & 1 ? kc.z : kc.x, o = q & 1 ? kc.w : kc.y;
        return as_v8h(make_uint4(pk_fma((r.x & m) | c, f, o), pk_fma(((r.x >> 8) & m) | c, f, o), pk_fma((r.y & m) | c, f, o),
                                 pk_fma(((r.y >> 8) & m) | c, f, o)));
    }
};

template <>
struct GpD<LE_TYPE_Q5_K> {
    uint4 nh;
    uint2 nq[2], qh[2];
    u32 scw, sc1, live;
    le_v8h b2;
    float d, dm;
    uint2 raw[2];
    uint4 kc;
    __device__ __forceinline__ void head(const u8 *rs, int hs) {
        nh = *(const uint4 *)rs;
        nq[0] = *(const uint2 *)(rs + 16 + 8 * hs);
        nq[1] = *(const uint2 *)(rs + 32 + 8 * hs);
    }
    __device__ __forceinline__ void prep(int h) {
        if (h == 0) {
            d = h2f(nh.x & 0xFFFFu);
            live = d == 0.f ? 0u : ~0u;
            scw = nh.y & 0x3F3F3F3Fu & live;
            sc1 = ((nh.w & 0x0F0F0F0Fu) | ((nh.y >> 2) & 0x30303030u)) & live;
            qh[0] = nq[0];
            qh[1] = nq[1];
            const u32 m0 = nh.z & 0x3F3F3F3Fu, m1 = ((nh.w >> 4) & 0x0F0F0F0Fu) | ((nh.z >> 2) & 0x30303030u);
            b2 = as_v8h(make_uint4(pk_add(h1024_02(m0), 0xE400E400u), pk_add(h1024_13(m0), 0xE400E400u),
                                   pk_add(h1024_02(m1), 0xE400E400u), pk_add(h1024_13(m1), 0xE400E400u)));
            dm = -h2f(nh.x >> 16);
        } else {
            scw = sc1;
        }
    }
    __device__ __forceinline__ void fetch(const u8 *rs, int q, int hs) {
        if ((q & 1) == 0) raw[(q >> 1) & 1] = *(const uint2 *)(rs + 48 + 32 * (q >> 2) + 16 * ((q >> 1) & 1) + 8 * hs);
    }
    __device__ __forceinline__ le_v8h frag(int q, int h, u32, u32, u32) {
        const int g = q >> 2, G = 2 * h + g, hi = q & 1, c1 = (q >> 1) & 1;
        if ((q & 3) == 0) {
            const u32 slo = pk_add(h1024_dup(scw, 2 * g), 0xE400E400u), shi = pk_add(h1024_dup(scw, 2 * g + 1), 0xE400E400u);
            kc = make_uint4(slo, pk_mul(slo, 0xE400E400u), shi, pk_mul(shi, 0xE400E400u));
        }
        const uint2 r = raw[c1], w = qh[c1];
        const u32 x = and_or(hi ? r.x >> 4 : r.x, 0x0F0F0F0Fu, ((w.x >> (2 * G + hi)) << 4) & 0x10101010u);
        const u32 y = and_or(hi ? r.y >> 4 : r.y, 0x0F0F0F0Fu, ((w.y >> (2 * G + hi)) << 4) & 0x10101010u);
        const u32 f = hi ? kc.z : kc.x, o = hi ? kc.w : kc.y;
        return as_v8h(make_uint4(pk_fma(h1024_02(x), f, o), pk_fma(h1024_13(x), f, o), pk_fma(h1024_02(y), f, o), pk_fma(h1024_13(y), f, o)));
    }
};

/* direct-to-LDS load, scalar base + per-lane 32-bit offset (gq_lds_dma16) */
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void gp_lds_dma16(const u8 *base, u32 off, u32 lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds_addr) : "memory", "m0");
}
#pragma clang diagnostic pop

template <int TY, int TM, bool GR, bool TB = false> /* TB: grouped form over a pointer table */
__device__ __forceinline__ void gp_body(const GqArgs &a, const u8 *ws) {
    using F = GqF<TY>;
    constexpr int SLOT = gp_slot<TY>(), N16 = SLOT / 16;
    constexpr int TN = 2, WN = 4, BM = 32 * TM, BN = 256;
    constexpr int WB = BN * SLOT, AB = BM * 256, SBYTES = 2 * TM * F::SREC; /* bytes of a weight / activation step slot, sum records */
    constexpr int NA = AB / 4096;                                            /* activation loads per thread and step */
    static_assert((size_t)3 * WB + 2 * AB >= (size_t)32 * (BN + 8) * 4, "output staging");
    extern __shared__ uint4 smem[];
    u8 *lds = (u8 *)smem, *Aring = lds + 3 * WB, *Sl = Aring + 2 * AB;

    const int K = a.cols, nsb = K >> 8;
    const int NTR1 = (a.rows + BN - 1) / BN, NTR = GR && a.dual ? 2 * NTR1 : NTR1, MT = GR ? a.maxt : (a.m + BM - 1) / BM;
    const int id = blockIdx.x, j = id >> 3; /* block order: gq_body */
    const int mt = NTR >= 8 ? j % MT : id / NTR, nt = NTR >= 8 ? (j / MT) * 8 + (id & 7) : id % NTR;
    if (nt >= NTR || mt >= MT) return;
    const bool second = nt >= NTR1;
    const int nb = (second ? nt - NTR1 : nt) * BN, nbw = min(nb, a.rows - BN), mb = mt * BM; /* rows nbw .. are computed, nb .. stored */
    int M = a.m, pair0 = 0;
    const u8 *Wsrc = a.w;
    if constexpr (GR) {
        int sl;
        if (!le_tile_of(a.off, a.nslot, a.bm, mt, sl, pair0)) return;
        M = mb + min(BM, a.off[sl + 1] - pair0);
        Wsrc = TB ? (second ? a.ptrs2 : a.ptrs)[sl] : (second ? a.w2 : a.w) + (size_t)sl * a.w_slot_bytes;
        if (TB && ((size_t)Wsrc & 15)) return; /* left to le_gqu_* */
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, hs = lane >> 5;
    const u32 rb = (u32)nsb * F::SBB;
    const int sb0 = blockIdx.y * (nsb / a.ksplit), sb1 = sb0 + nsb / a.ksplit, s0 = 2 * sb0, nstep = 2 * sb1;
    const u8 *Ag = ws + (size_t)(mb / 32) * (K / 16) * 1024;
    const u8 *Sg = ws + gq_s_off(a.mp, K) + ((size_t)(mb / 32) + (wave % TM)) * nsb * F::SREC;
    const float *tsc = (const float *)(ws + gq_t_off(a.mp, K, F::SREC));

    /* Weights of the wave's 64 rows: load i of the wave fills bytes 1024 i .. of its part of a slot, rows
     * without padding (an odd number of 16-byte pieces each). The last row tile starts early enough to be
     * whole: the caller has rows >= 256. */
    u32 wd[N16];
#pragma unroll
    for (int i = 0; i < N16; i++) {
        const int c = lane + 64 * i, row = c / N16, k = c - row * N16;
        wd[i] = (u32)row * rb + F::goff(k, 0);
    }
    u8 *wlds = lds + 64 * wave * SLOT;
    const u32 wlds0 = gq_lds_addr(lds) + (u32)(64 * SLOT) * (u32)wave;
    const u8 *wrow = Wsrc + (size_t)(nbw + 64 * wave) * rb;
    auto wdma = [&](int s_, int h, u32 slot, int i0, int i1) { /* loads i0 .. i1 of step s_ (parity h) into the step slot at LDS offset slot */
        /* past the slice's end the last step again */
        const u8 *w0 = wrow + (size_t)(min(s_, nstep - 2 + h) >> 1) * F::SBB + 64 * h;
#pragma unroll
        for (int i = i0; i < i1; i++) gp_lds_dma16(w0, wd[i], __builtin_amdgcn_readfirstlane(wlds0 + slot + 1024u * i));
    };
    /* activations of step s_ (parity h); grouped form: lanes of tokens past the tile's last pair re-read
     * token 0's (their rows are never stored), so a sparse tile fetches fewer lines */
    u32 xo[GR ? NA : 1];
    if constexpr (GR) {
#pragma unroll
        for (int i = 0; i < NA; i++) {
            const int c = tid + 256 * i, tl = c >> 9, off = c & 511;
            const bool ok = mb + 32 * tl + (off & 31) < M;
            xo[i] = (ok ? (u32)tl * (u32)(K / 16) * 1024u : 0u) + 16u * (u32)(ok ? off : off & ~31);
        }
    }
    const u32 alds = gq_lds_addr(Aring) + 1024u * (u32)wave, slds = gq_lds_addr(Sl) + 1024u * (u32)(wave % TM);
    auto dma = [&](int s_, int h, int p) { /* quarter p of a step's loads */
        const u8 *x0 = Ag + (size_t)min(s_, nstep - 2 + h) * 8192;
#pragma unroll
        for (int i = p * NA / 4; i < (p + 1) * NA / 4; i++) {
            const u32 la = __builtin_amdgcn_readfirstlane(alds + (u32)(h * AB) + 4096u * i);
            if constexpr (GR)
                gp_lds_dma16(x0, xo[i], la);
            else
                gp_lds_dma16(x0 + (size_t)(i >> 1) * (K / 16) * 1024 + 4096 * (i & 1), 16u * (u32)tid, la);
        }
    };
    auto dmas = [&](int sb) { /* sum records of super-block sb, one 1 KB tile per wave */
        gp_lds_dma16(Sg + (size_t)min(sb, sb1 - 1) * F::SREC, 16u * (u32)lane, __builtin_amdgcn_readfirstlane(slds + (u32)((sb & 1) * TM * F::SREC)));
    };

    le_v16f acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int k = 0; k < TN; k++) acc[i][k] = (le_v16f){};
    GpD<TY> D[TN];
    float unit[TN], ratio[TN];
#pragma unroll
    for (int k = 0; k < TN; k++) unit[k] = ratio[k] = 1.f;
    const u8 *rs[TN];
#pragma unroll
    for (int k = 0; k < TN; k++) rs[k] = wlds + (32 * k + n) * SLOT;
    auto head = [&](u32 slot) {
#pragma unroll
        for (int k = 0; k < TN; k++) D[k].head(rs[k] + slot, hs);
    };
    auto prep = [&](int h) {
#pragma unroll
        for (int k = 0; k < TN; k++) {
            D[k].prep(h);
            if (h == 0) { /* a new super-block scale: the running sums go into its units (a zero scale keeps the old ones) */
                ratio[k] = D[k].d == 0.f ? 1.f : unit[k] * __builtin_amdgcn_rcpf(D[k].d);
                unit[k] = D[k].d == 0.f ? unit[k] : D[k].d;
                D[k].dm *= __builtin_amdgcn_rcpf(unit[k]);
            }
        }
    };
    auto fetch = [&](u32 slot, int q) {
#pragma unroll
        for (int k = 0; k < TN; k++) D[k].fetch(rs[k] + slot, q, hs);
    };
    le_v8h A[TM], B[2][TN];
    le_v16f d2 = {};
    constexpr int SV = 4; /* other VALU instructions per MFMA */
    auto aload = [&](int h, int q, int i) { /* activation fragment i of position q: its 16-value chunk of the step */
        const int c = (q & 4) | ((q & 1) << 1) | ((q >> 1) & 1);
        A[i] = as_v8h(*(const uint4 *)(Aring + h * AB + i * 8192 + c * 1024 + lane * 16));
    };
    /* the decoders' masks in registers the compiler cannot see through, so (x & m) | c becomes one
     * v_and_or_b32 (which cannot carry literals); the inline form costs a wait state per use */
    u32 cmlo = 0x000F000Fu, cmhi = 0x00F000F0u, c1024 = 0x64006400u;
    __asm__("" : "+v"(cmlo), "+v"(cmhi), "+s"(c1024));
    auto frag = [&](int h, int q) {
#pragma unroll
        for (int k = 0; k < TN; k++) B[q & 1][k] = D[k].frag(q, h, cmlo, cmhi, c1024);
    };

    u32 wc = 0, wn1 = WB, wn2 = 2 * WB; /* weight slots of this step and the next two */
    wdma(s0, 0, wc, 0, N16);
#pragma unroll
    for (int p = 0; p < 4; p++) dma(s0, 0, p);
    dmas(sb0);
    wdma(s0 + 1, 1, wn1, 0, N16);
    gq_vm_wait<N16>();
    __syncthreads();
    dma(s0 + 1, 1, 0);
    head(wc);
    fetch(wc, 0);
#pragma unroll
    for (int i = 0; i < TM; i++) aload(0, 0, i);
    fetch(wc, 1);
    prep(0);
    frag(0, 0);
    for (int sb = sb0; sb < sb1; sb++) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int s = 2 * sb + h;
#pragma unroll
            for (int q = 0; q < 8; q++) {
                const int h1 = q == 7 ? h ^ 1 : h, q1 = (q + 1) & 7, q2 = (q + 2) & 7;
                if (q == 7) {
                    __builtin_amdgcn_sched_barrier(0);
                    /* the step's last activation fragments are in registers, the next step's have
                     * landed (younger: the weight loads issued after them) */
                    gq_vm_wait<N16>();
                    gq_barrier();
                    __builtin_amdgcn_sched_barrier(0);
                }
                /* a few loads at a time: a burst of them holds up the wave's instructions, MFMAs among them */
                if (q == 7) dma(s + 2, h, 0);
                if (q < 3) dma(s + 1, h ^ 1, q + 1);
                if (q == 2 && h == 0) dmas(sb + 1);
                if (q >= 3 && q < 6) wdma(s + 2, h, wn2, (q - 3) * N16 / 3, (q - 2) * N16 / 3);
                if (q == 6) { /* the next step's weights have landed: younger are its activations, sum records and the weights after it */
                    if (h == 0) gq_vm_wait<NA + N16 + 1>();
                    else gq_vm_wait<NA + N16>();
                    if (h == 1) head(wn1);
                }
                fetch(q >= 6 ? wn1 : wc, q2);
                if (h == 0 && q == 0) {
#pragma unroll
                    for (int k = 0; k < TN; k++)
#pragma unroll
                        for (int i = 0; i < TM; i++)
#pragma unroll
                            for (int e = 0; e < 16; e++) acc[i][k][e] *= ratio[k];
                }
                /* offset term -dmin sum_j m_j S_j, in units, of one tile per position: its MFMA at position
                 * g - 1 = tile of the super-block, added one position later */
                const int g = 8 * h + q;
                if (g >= 2 && g - 2 < TM * TN) {
                    const int i = (g - 2) / TN, k = (g - 2) % TN;
#pragma unroll
                    for (int e = 0; e < 16; e++) acc[i][k][e] = __builtin_fmaf(D[k].dm, d2[e], acc[i][k][e]);
                }
                if (g >= 1 && g - 1 < TM * TN) {
                    const int i = (g - 1) / TN, k = (g - 1) % TN;
                    const le_v8h a2 = as_v8h(*(const uint4 *)(Sl + ((sb & 1) * TM + i) * 1024 + lane * 16));
                    d2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a2, D[k].b2, (le_v16f){}, 0, 0, 0);
                }
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int k = 0; k < TN; k++) acc[i][k] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[i], B[q & 1][k], acc[i][k], 0, 0, 0);
#pragma unroll
                for (int i = 0; i < TM; i++) aload(h1, q1, i); /* each once its MFMAs have been issued: into the same registers */
                if (q == 7) prep(h ^ 1);
                frag(h1, q1);
                /* MFMAs evenly among the position's other instructions */
#pragma unroll
                for (int i = 0; i < TM; i++) {
#pragma unroll
                    for (int k = 0; k < TN; k++) {
                        if (g == 0) __builtin_amdgcn_sched_group_barrier(0x002, 17, 0); /* the rescaling */
                        else __builtin_amdgcn_sched_group_barrier(0x002, SV, 0);
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    }
                    __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            const u32 w = wc;
            wc = wn1;
            wn1 = wn2;
            wn2 = w;
        }
    }
    gq_vm_wait<0>(); /* no load may still be writing LDS */
#pragma unroll
    for (int k = 0; k < TN; k++) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][k][e] *= unit[k];
    }
    gq_store<1, WN, TM, TN, GR, 3 * WB + 2 * AB, true>(a, lds, tsc, acc, M, mb, nbw, pair0, second, nb);
}

#define LE_GQX(TY, SK) \
    extern "C" __global__ void __launch_bounds__(256) le_gq_xprep_##TY(GqArgs a, u8 *ws) { gq_xprep_body<SK>(a, ws); } \
    extern "C" __global__ void __launch_bounds__(256) le_gq_xprepg_##TY(GqArgs a, u8 *ws) { gq_xprep_body<SK, true>(a, ws); } \
    extern "C" __global__ void __launch_bounds__(256) le_gq_xprepw_##TY(GqArgs a, u8 *ws) { gq_xprepw_body<SK>(a, ws); }
/* two code objects, compiled in parallel: the five types of the reference's mmq kernels, and the
 * four formats added beside them (LE_GQ_SET=2) */
#if LE_GQ_SET == 2
LE_GQX(2, 0) LE_GQX(11, 0) LE_GQX(13, 1) LE_GQX(22, 0)
#else
LE_GQX(8, 0) LE_GQX(12, 1) LE_GQX(14, 0) LE_GQX(16, 0) LE_GQX(18, 0)
#endif

/* Sum of the K slices' partial results: y[e] = part[0][e] + part[1][e] + ... in slice order
 * (deterministic, unlike atomic adds). */
#if LE_GQ_SET != 2
extern "C" __global__ void __launch_bounds__(256) le_gq_ksum(GqArgs a) {
    const size_t n = (size_t)a.m * a.rows, st = (size_t)gridDim.x * blockDim.x;
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int ks = a.ksplit;
    if ((n & 3) == 0 && ((size_t)a.y & 15) == 0) { /* part is 256-byte aligned in the workspace */
        const size_t n4 = n / 4;
        const float4 *p = (const float4 *)a.part;
        for (; i < n4; i += st) {
            float4 s = p[i];
            for (int q = 1; q < ks; q++) {
                const float4 v = p[q * n4 + i];
                s.x += v.x;
                s.y += v.y;
                s.z += v.z;
                s.w += v.w;
            }
            ((float4 *)a.y)[i] = s;
        }
    } else {
        for (; i < n; i += st) {
            float s = a.part[i];
            for (int q = 1; q < ks; q++) s += a.part[q * n + i];
            a.y[i] = s;
        }
    }
}

#endif

#define LE_GQ_(TY, WM, WN, TM, TN)                                                                                     \
    extern "C" __global__ void __launch_bounds__(WM * WN * 64) le_gq_##TY##_w##WM##WN##_t##TM##TN(GqArgs a, const u8 *ws) { \
        gq_body<TY, WM, WN, TM, TN, false, 2>(a, ws, blockIdx.x);                                                                  \
    }
#define LE_GQG_(TY, WM, WN, TM, TN)                                                                                     \
    extern "C" __global__ void __launch_bounds__(WM * WN * 64) le_gqg_##TY##_w##WM##WN##_t##TM##TN(GqArgs a, const u8 *ws) { \
        gq_body<TY, WM, WN, TM, TN, true, 2>(a, ws, blockIdx.x);                                                                     \
    }
/* one wave per SIMD is resident (LDS), but 256 registers: with 512 the accumulators go to the
 * accumulation registers, which the rescaling cannot reach without moves (393 reads a super-block) */
#define LE_GP_REGS __attribute__((amdgpu_waves_per_eu(2, 2)))
#define LE_GP_(TY, TM)                                                                                                  \
    extern "C" __global__ void __launch_bounds__(256) LE_GP_REGS le_gp_##TY##_t##TM(GqArgs a, const u8 *ws) { gp_body<TY, TM, false>(a, ws); } \
    extern "C" __global__ void __launch_bounds__(256) LE_GP_REGS le_gpg_##TY##_t##TM(GqArgs a, const u8 *ws) { gp_body<TY, TM, true>(a, ws); } \
    extern "C" __global__ void __launch_bounds__(256) LE_GP_REGS le_gpgt_##TY##_t##TM(GqArgs a, const u8 *ws) { gp_body<TY, TM, true, true>(a, ws); }
#define LE_GQU_(TY, WM, WN, TM, TN) \
    extern "C" __global__ void __launch_bounds__(WM * WN * 64) le_gqu_##TY##_w##WM##WN##_t##TM##TN(GqArgs a, const u8 *ws) { gqu_body<TY, WM, WN, TM, TN>(a, ws); }
#define LE_GP(TY) LE_GP_(TY, 4) LE_GP_(TY, 2) LE_GQU_(TY, 1, 8, 4, 1) LE_GQU_(TY, 1, 8, 2, 1)
#define LE_GQ(TY) LE_GQ_(TY, 1, 4, 1, 2) LE_GQ_(TY, 1, 4, 2, 2) LE_GQ_(TY, 1, 4, 4, 2) LE_GQ_(TY, 2, 2, 2, 2) \
    LE_GQ_(TY, 1, 8, 2, 1) LE_GQ_(TY, 1, 8, 4, 1) LE_GQ_(TY, 1, 8, 1, 1) LE_GQ_(TY, 1, 4, 2, 1) LE_GQ_(TY, 1, 4, 1, 1) LE_GQ_(TY, 1, 4, 4, 1) LE_GQG_(TY, 1, 8, 2, 1) LE_GQG_(TY, 1, 8, 4, 1) LE_GQG_(TY, 2, 2, 2, 2) LE_GQG_(TY, 1, 8, 1, 1) LE_GQG_(TY, 1, 4, 1, 1)
#if LE_GQ_SET == 2
LE_GQ(2) LE_GQ(11) LE_GQ(13) LE_GQ(22)
LE_GP(13)
#else
LE_GQ(8) LE_GQ(12) LE_GQ(14) LE_GQ(16) LE_GQ(18)
LE_GP(12)
LE_GQ_(12, 2, 4, 2, 2) LE_GQ_(12, 2, 4, 2, 1)
#endif
