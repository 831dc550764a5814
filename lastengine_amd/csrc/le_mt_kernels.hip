/* Few-token quantized GEMM for every type (gfx950): Y[t, r] = W[r, :] . X[t, :] for t < m <= 16 tokens, the
 * speculative-verify shape of mmq*_<ty> (src/cuda/kernels.cu:965-1235; CPU twin cpu_ref::matmat,
 * src/cpu_ref.rs:266-276). One pass over the weights, the tokens as the rows of
 * v_mfma_f32_16x16x32_f16.
 *
 * Operands. A (16 x 32): the 16 MFMA rows hold, for T = 8, the high halves of eight tokens (rows 0-7) and
 * their low halves (rows 8-15); for T = 4 rows 0-3 and 4-7 (the rest zero); for T = 16 the tokens
 * rounded once. Each token's 256-value super-block is scaled by the power of two that puts its largest
 * magnitude in [512, 1024); high half = fp16(x), low half = fp16((x - high) 2^11), together about
 * 2^-22 per value (T = 16: 2^-11, as in the larger GEMMs). B (32 x 16): 16 weight rows, the 32
 * values of one sub-block as exact fp16 codes:
 *   Q4_K, Q5_K       sc_j q, offset term sum_j m_j S_j by one more MFMA per super-block (S_j: sums of the
 *                    rounded halves, themselves split in two)          (src/quant.rs:72-95)
 *   Q6_K             sc (ql nibble) and 16 sc (qh - 2), two MFMAs (q - 32 times sc does not fit 11 bits)  (:96-112)
 *   Q3_K, IQ2_XXS, IQ3_XXS, IQ2_S   scale times code, as in the larger GEMM   (:113-167)
 *   Q8_0, Q4_0       q, the block scale in the per-sub-block epilogue         (:64-71)
 * Per super-block: y += d 2^e D.
 *
 * Work. A block of 8 waves builds the fp16 images of its K slice in LDS once (no pre-pass launch) and loops
 * over row tiles of 16: KW waves split the slice's super-blocks of one tile (summed through LDS), 8 / KW
 * tiles run side by side. Each wave streams its tile's super-blocks one item ahead in registers and
 * stages them in a wave-private LDS buffer (rows of an odd number of 16-byte slots), as the decode
 * matvec does. blockIdx.y: K slices whose partial results le_gq_ksum adds in slice order (only where the
 * images of all of K do not fit the LDS).
 *
 * Grouped form le_mtg_* (the MoE layer's few tokens an expert; grouped mm, src/cuda/kernels.cu:679-719): ng
 * blocks share a tile of up to T pairs of one slot, rounded once, and optionally gate and up in one launch. It
 * has no pre-pass (a launch and a pass over the images less) and no padding to 32 pairs; figures where it is chosen.
 *
 * It replaces, below nine tokens, vector kernels that unpack every weight for each pair of tokens, and to 16
 * tokens the larger GEMM. Measured at 4 / 8 / 16 tokens: Q6_K 4096 x 14336 67.0 -> 24.8, 124 -> 22.2, 30.6 ->
 * 29.7 us; Q8_0 32000 x 4096 69.8 -> 32.4, 94.3 -> 34.2, 51.7 -> 36.0; IQ2_XXS 14336 x 4096 34.3 -> 16.1,
 * 47.9 -> 18.3, 27.1 -> 19.9. Bound by the decoding (Q6_K: about 240 VALU instructions a super-block, Q4_K 156) and,
 * for small matrices, by each block's image build (2 -> 8 tokens of Q4_0 4096 x 4096: 7.6 -> 10.5 us). */
#include "le_f16_frag.h"
#include "le_mt_layout.h"

typedef float le_v4f __attribute__((ext_vector_type(4)));

struct MtArgs {
    const u8 *w;
    const float *x;
    float *y, *part; /* part: [slices][m][rows], or null with one slice */
    int rows, cols, m, kw;
    /* grouped form: slot s multiplies weight ptrs[s] (or w + s * w_slot_bytes) with the rows in_idx[i] of x (with
     * up: silu(x) * up) of its pairs i in off[s] .. off[s+1], writing output rows out_idx[i]; dual: a second weight
     * set (ptrs2 or w2, same shape) into y2 */
    const u8 *const *ptrs;
    unsigned long long w_slot_bytes;
    const int *off, *in_idx, *out_idx;
    int nslot, cus, units, ng, dual; /* units: groups of row tiles; ng: blocks that share them under an even routing */
    const u8 *const *ptrs2;
    const u8 *w2;
    float *y2;
    const float *up;
};

/* staged super-blocks: CPS 16-byte chunks, chunk c read from byte goff(c) */
template <int TY>
struct MtF;
template <>
struct MtF<LE_TYPE_Q4_K> {
    static constexpr int CPS = 9, SBB = 144;
    __device__ static int goff(int c) { return 16 * c; }
};
template <>
struct MtF<LE_TYPE_Q5_K> {
    static constexpr int CPS = 11, SBB = 176;
    __device__ static int goff(int c) { return 16 * c; }
};
template <>
struct MtF<LE_TYPE_Q6_K> { /* bytes 0-207, then 194-209 (d in the last two) */
    static constexpr int CPS = 14, SBB = 210;
    __device__ static int goff(int c) { return c == 13 ? 194 : 16 * c; }
};
template <>
struct MtF<LE_TYPE_Q3_K> { /* bytes 0-95, then 94-109 (scales from its byte 2, d in the last two) */
    static constexpr int CPS = 7, SBB = 110;
    __device__ static int goff(int c) { return c == 6 ? 94 : 16 * c; }
};
template <>
struct MtF<LE_TYPE_IQ2_S> { /* bytes 0-79, then 66-81 (qh, scales) */
    static constexpr int CPS = 6, SBB = 82;
    __device__ static int goff(int c) { return c == 5 ? 66 : 16 * c; }
};
template <>
struct MtF<LE_TYPE_IQ2_XXS> { /* from byte 2, then bytes 0-15 (d) */
    static constexpr int CPS = 5, SBB = 66;
    __device__ static int goff(int c) { return c < 4 ? 2 + 16 * c : 0; }
};
template <>
struct MtF<LE_TYPE_IQ3_XXS> {
    static constexpr int CPS = 7, SBB = 98;
    __device__ static int goff(int c) { return c < 6 ? 2 + 16 * c : 0; }
};
template <>
struct MtF<LE_TYPE_Q8_0> {
    static constexpr int CPS = 17, SBB = 272;
    __device__ static int goff(int c) { return 16 * c; }
};
template <>
struct MtF<LE_TYPE_Q4_0> {
    static constexpr int CPS = 9, SBB = 144;
    __device__ static int goff(int c) { return 16 * c; }
};

/* 8 bytes at byte b of a staged super-block (LDS, 16-byte aligned) that lie in `words` words: 2, or 3 from the
 * middle of the first. No word past them is read: the last group of the last staged row ends the block's LDS. */
__device__ __forceinline__ uint2 mt_lds8(const u8 *sb, int b, int words) {
    const u32 *w = (const u32 *)(sb + (words == 3 ? b - 2 : b));
    const u32 w0 = w[0], w1 = w[1];
    return words == 3 ? make_uint2(__builtin_amdgcn_alignbit(w1, w0, 16), __builtin_amdgcn_alignbit(w[2], w1, 16)) : make_uint2(w0, w1);
}
__device__ __forceinline__ le_v8h mt_codes(u32 x, u32 y, u32 bias) { /* bytes minus (bias - 1024) as halves */
    return as_v8h(make_uint4(pk_add(h1024_02(x), bias), pk_add(h1024_13(x), bias), pk_add(h1024_02(y), bias), pk_add(h1024_13(y), bias)));
}
__device__ __forceinline__ le_v8h mt_codes_sc(u32 x, u32 y, u32 bias, u32 sc) {
    return as_v8h(make_uint4(pk_mul(pk_add(h1024_02(x), bias), sc), pk_mul(pk_add(h1024_13(x), bias), sc),
                             pk_mul(pk_add(h1024_02(y), bias), sc), pk_mul(pk_add(h1024_13(y), bias), sc)));
}
/* bytes times sc, exact: (1024 + u) sc - 1024 sc in one rounding; 1024 sc has to be finite (sc < 64) */
__device__ __forceinline__ le_v8h mt_codes_fma(u32 x, u32 y, u32 sc) {
    const u32 k = pk_mul(sc, 0xE400E400u);
    return as_v8h(make_uint4(pk_fma(h1024_02(x), sc, k), pk_fma(h1024_13(x), sc, k), pk_fma(h1024_02(y), sc, k), pk_fma(h1024_13(y), sc, k)));
}
__device__ __forceinline__ le_v8h mt_grid(uint4 g, uint4 m, u32 f) {
    return as_v8h(make_uint4(pk_mul(g.x, f) ^ m.x, pk_mul(g.y, f) ^ m.y, pk_mul(g.z, f) ^ m.z, pk_mul(g.w, f) ^ m.w));
}

/* y += the 16 x 16 products of one super-block: row sb of 16 weight rows (lane: row n = lane % 16, 8-value
 * group g = lane / 16 of every sub-block), image a (fragment (j, g) of row m at slot (4 j + g) RS + m), sums
 * fragment at slot 32 RS + g RS + m (g < 2), scales st of the four MFMA rows 4 g ... */
template <int TY, int R, int RS>
__device__ __forceinline__ void mt_sb(const u8 *sb, const uint4 *a, int lane, float4 st, const u8 *tab, le_v4f &y) {
    const int g = lane >> 4, m = lane & 15;
    const u32 *w32 = (const u32 *)sb;
    /* the super-block's LDS reads all first: read where they are used, each MFMA waited out one of them
     * (about 1 us an item with two waves on a SIMD) */
    uint4 Af[8];
#pragma unroll
    for (int j = 0; j < 8; j++) Af[j] = a[(4 * j + g) * RS + (m & (R - 1))]; /* R = 8: MFMA rows 8-15 repeat 0-7, unused */
    auto A = [&](int j) { return as_v8h(Af[j]); };
    auto mm = [](le_v8h x, le_v8h w, le_v4f d) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(x, w, d, 0, 0, 0); };
    le_v4f D = {0.f, 0.f, 0.f, 0.f};
    float d;
    if constexpr (TY == LE_TYPE_Q4_K || TY == LE_TYPE_Q5_K) {
        constexpr bool Q5 = TY == LE_TYPE_Q5_K;
        const uint4 hd = *(const uint4 *)sb;
        const u32 sc[2] = {hd.y & 0x3F3F3F3Fu, (hd.w & 0x0F0F0F0Fu) | ((hd.y >> 2) & 0x30303030u)};
        uint2 qh = make_uint2(0, 0), qv[4];
        if constexpr (Q5) qh = *(const uint2 *)(sb + 16 + 8 * g);
#pragma unroll
        for (int G = 0; G < 4; G++) qv[G] = *(const uint2 *)(sb + (Q5 ? 48 : 16) + 32 * G + 8 * g);
        const le_v8h S = as_v8h(a[(32 + (g & 1)) * RS + (m & (R - 1))]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int G = 0; G < 4; G++) {
            const uint2 q = qv[G];
#pragma unroll
            for (int hi = 0; hi < 2; hi++) {
                const int j = 2 * G + hi;
                u32 x = (q.x >> (4 * hi)) & 0x0F0F0F0Fu, z = (q.y >> (4 * hi)) & 0x0F0F0F0Fu;
                if constexpr (Q5) {
                    x |= ((qh.x >> j) & 0x01010101u) << 4;
                    z |= ((qh.y >> j) & 0x01010101u) << 4;
                }
                D = mm(A(j), mt_codes_fma(x, z, pk_add(h1024_dup(sc[j >> 2], j & 3), 0xE400E400u)), D);
            }
        }
        const u32 m0 = hd.z & 0x3F3F3F3Fu, m1 = ((hd.w >> 4) & 0x0F0F0F0Fu) | ((hd.z >> 2) & 0x30303030u);
        /* K positions 16-31 of the offset MFMA: zero mins */
        const u32 k2 = g < 2 ? ~0u : 0u;
        const le_v4f O = mm(S, mt_codes(m0 & k2, m1 & k2, 0xE400E400u), (le_v4f){0.f, 0.f, 0.f, 0.f});
        d = h2f(hd.x & 0xFFFFu);
        const float dm = h2f(hd.x >> 16);
#pragma unroll
        for (int e = 0; e < 4; e++) D[e] = d * D[e] - dm * O[e];
        d = 1.f;
    } else if constexpr (TY == LE_TYPE_Q6_K) {
        /* value 128 hn + 32 s + l: ql byte 64 hn + 32 (s & 1) + l (nibble s / 2), qh byte 32 hn + l bits 2s, scale 8 hn + 2 s + l / 16 */
        const uint4 scv = *(const uint4 *)(sb + 192);
        const u32 scw[4] = {scv.x, scv.y, scv.z, scv.w}, dw = *(const u32 *)(sb + 220);
        uint2 qlv[4], qhv[2];
#pragma unroll
        for (int i = 0; i < 4; i++) qlv[i] = *(const uint2 *)(sb + 32 * i + 8 * g);
#pragma unroll
        for (int hn = 0; hn < 2; hn++) qhv[hn] = *(const uint2 *)(sb + 128 + 32 * hn + 8 * g);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int hn = 0; hn < 2; hn++) {
            const uint2 qh = qhv[hn];
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const uint2 ql = qlv[2 * hn + (s & 1)];
                const u32 w = scw[2 * hn + (s >> 1)] ^ 0x80808080u; /* scales 8 hn + 2 s, + 1 in bytes 2 (s & 1), + 1 */
                /* scale / 16, from the byte under the exponent of 64: 1024 times the scale itself can pass 65504 */
                const u32 sc = pk_add(__builtin_amdgcn_perm(0x54545454u, w, (s & 1 ? 0x04020402u : 0x04000400u) + (u32)(g >> 1) * 0x00010001u), 0xD480D480u);
                const le_v8h av = A(4 * hn + s);
                D = mm(av, mt_codes_fma((ql.x >> (4 * (s >> 1))) & 0x0F0F0F0Fu, (ql.y >> (4 * (s >> 1))) & 0x0F0F0F0Fu, sc), D);
                const u32 hx = s < 2 ? qh.x << (4 - 2 * s) : qh.x >> (2 * s - 4), hy = s < 2 ? qh.y << (4 - 2 * s) : qh.y >> (2 * s - 4);
                D = mm(av, mt_codes_sc(hx & 0x30303030u, hy & 0x30303030u, 0xE420E420u, sc), D); /* 16 qh - 32 */
            }
        }
        d = 16.f * h2f(dw >> 16);
    } else if constexpr (TY == LE_TYPE_Q3_K) {
        const uint4 c6 = *(const uint4 *)(sb + 96);
        const u32 s0 = __builtin_amdgcn_alignbyte(c6.y, c6.x, 2), s1 = __builtin_amdgcn_alignbyte(c6.z, c6.y, 2), s2 = __builtin_amdgcn_alignbyte(c6.w, c6.z, 2);
        const uint2 hm = *(const uint2 *)(sb + 8 * g), qv[2] = {*(const uint2 *)(sb + 32 + 8 * g), *(const uint2 *)(sb + 64 + 8 * g)};
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int hn = 0; hn < 2; hn++) {
            const uint2 qs = qv[hn];
            /* scales 8 hn + i: low 4 bits nibble hn of byte i, bits 4-5 from byte 8 + i % 4 */
            const u32 v[2] = {((s0 >> (4 * hn)) & 0x0F0F0F0Fu) | (((s2 >> (4 * hn)) & 0x03030303u) << 4),
                              ((s1 >> (4 * hn)) & 0x0F0F0F0Fu) | (((s2 >> (4 * hn + 2)) & 0x03030303u) << 4)};
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const u32 sc = pk_add(h1024_dup((v[s >> 1] >> (16 * (s & 1) + 8 * (g >> 1))) & 255u, 0), 0xE420E420u); /* scale - 32 */
                const u32 x = ((qs.x >> (2 * s)) & 0x03030303u) | (((hm.x >> (4 * hn + s)) & 0x01010101u) << 2);
                const u32 z = ((qs.y >> (2 * s)) & 0x03030303u) | (((hm.y >> (4 * hn + s)) & 0x01010101u) << 2);
                D = mm(A(4 * hn + s), mt_codes_sc(x, z, 0xE404E404u, sc), D);
            }
        }
        d = h2f(c6.w >> 16);
    } else if constexpr (TY == LE_TYPE_IQ2_S) {
        u32 w[24]; /* the index, sign, high-bit and scale words */
#pragma unroll
        for (int i = 0; i < 24; i++) w[i] = i == 18 || i == 19 ? 0u : w32[i];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint4 gv[4], sv[4];
            u32 f[4];
#pragma unroll
            for (int i = 0; i < 4; i++) { /* index byte 2 + 4 j + g, sign byte 34 + 4 j + g (2 mod 4 aligned) */
                const int j = 4 * h + i;
                const u32 q = __builtin_amdgcn_alignbit(w[j + 1], w[j], 16), sg = __builtin_amdgcn_alignbit(w[9 + j], w[8 + j], 16);
                const u32 qh = (w[20 + h] >> (8 * i)) & 255u, sc = (w[22 + h] >> (8 * i + 4 * (g >> 1))) & 15u;
                const u32 gi = ((q >> (8 * g)) & 255u) | ((qh << (8 - 2 * g)) & 0x300u);
                f[i] = pk_add(h1024_dup(2u * sc + 1u, 0), 0xE400E400u);
                gv[i] = *(const uint4 *)(tab + 16 * gi);
                sv[i] = *(const uint4 *)(tab + 16384 + 16 * ((sg >> (8 * g)) & 255u));
            }
#pragma unroll
            for (int i = 0; i < 4; i++) D = mm(A(4 * h + i), mt_grid(gv[i], sv[i], f[i]), D);
        }
        d = 0.125f * h2f(w[0] & 0xFFFFu);
    } else if constexpr (TY == LE_TYPE_IQ2_XXS || TY == LE_TYPE_IQ3_XXS) {
        constexpr bool I2 = TY == LE_TYPE_IQ2_XXS;
        const u8 *sgt = tab + (I2 ? 4096 : 2048);
        uint2 qv[8];
        u32 av[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            qv[j] = *(const uint2 *)(sb + 8 * j);
            av[j] = I2 ? qv[j].y : *(const u32 *)(sb + 64 + 4 * j);
        }
        const u32 dw = *(const u32 *)(sb + (I2 ? 64 : 96));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint4 gv[4], sv[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint2 q = qv[4 * h + i];
                sv[i] = *(const uint4 *)(sgt + 16 * ((av[4 * h + i] >> (7 * g)) & 127u));
                if constexpr (I2) {
                    gv[i] = *(const uint4 *)(tab + 16 * ((q.x >> (8 * g)) & 255u));
                } else {
                    const u32 iw = (g < 2 ? q.x : q.y) >> (16 * (g & 1));
                    const uint2 g0 = *(const uint2 *)(tab + 8 * (iw & 255u)), g1 = *(const uint2 *)(tab + 8 * ((iw >> 8) & 255u));
                    gv[i] = make_uint4(g0.x, g0.y, g1.x, g1.y);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const u32 f = pk_add(h1024_dup(2u * (av[4 * h + i] >> 28) + 1u, 0), 0xE400E400u);
                D = mm(A(4 * h + i), mt_grid(gv[i], sv[i], f), D);
            }
        }
        d = (I2 ? 0.125f : 0.25f) * h2f(dw & 0xFFFFu);
    } else { /* Q8_0, Q4_0: one scale per sub-block */
        constexpr bool Q8 = TY == LE_TYPE_Q8_0;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            uint2 qv[4];
            u32 dw[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int j = 4 * h + i, db = le_mt_byte(TY, j, 0) - 2; /* the scale: the low half of a word in even sub-blocks */
                dw[i] = j & 1 ? *(const u32 *)(sb + db - 2) >> 16 : *(const u32 *)(sb + db);
                qv[i] = mt_lds8(sb, le_mt_byte(TY, j, Q8 ? g : g & 1), le_mt_words(j));
            }
            __builtin_amdgcn_sched_barrier(0);
            le_v4f Dj[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                uint2 q = qv[i];
                if constexpr (Q8)
                    q = make_uint2(q.x ^ 0x80808080u, q.y ^ 0x80808080u);
                else
                    q = make_uint2((q.x >> (4 * (g >> 1))) & 0x0F0F0F0Fu, (q.y >> (4 * (g >> 1))) & 0x0F0F0F0Fu);
                Dj[i] = mm(A(4 * h + i), mt_codes(q.x, q.y, Q8 ? 0xE480E480u : 0xE408E408u), (le_v4f){0.f, 0.f, 0.f, 0.f});
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float dj = h2f(dw[i] & 0xFFFFu);
#pragma unroll
                for (int e = 0; e < 4; e++) D[e] = __builtin_fmaf(dj, Dj[i][e], D[e]);
            }
        }
        d = 1.f;
    }
    const float s4[4] = {st.x, st.y, st.z, st.w};
#pragma unroll
    for (int e = 0; e < 4; e++) y[e] = __builtin_fmaf(d * s4[e], D[e], y[e]);
}

/* largest of the wave's nonnegative values, uniform (DPP: no LDS round trips) */
__device__ __forceinline__ int mt_wave_max(int v) {
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true)); /* row_shr:1, 2, 4, 8 */
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false)); /* row_bcast:15, 31 */
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false));
    return __builtin_amdgcn_readlane(v, 63);
}
template <int CTRL>
__device__ __forceinline__ float mt_dpp_add(float v) {
    return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
/* sum over the lane's group of eight */
__device__ __forceinline__ float mt_sum8(float v) { return mt_dpp_add<0x141>(mt_dpp_add<0x4E>(mt_dpp_add<0xB1>(v))); } /* xor 1, xor 2, half-row mirror */

/* T tokens (GR: pairs of one slot) per pass, HL: as two halves */
template <int TY, int T, bool HL, bool GR>
__device__ __forceinline__ void mt_body(const MtArgs &a) {
    using F = MtF<TY>;
    constexpr bool OFS = TY == LE_TYPE_Q4_K || TY == LE_TYPE_Q5_K, AL = OFS; /* AL: 16-byte aligned weights */
    constexpr int R = HL ? 2 * T : T, RS = R + 1;              /* live MFMA rows; slots per fragment (odd: rows of the build's stores in distinct banks) */
    constexpr int IMG = (32 + (OFS ? 2 : 0)) * RS;             /* 16-byte slots of a super-block's image */
    static_assert(F::CPS == le_mt_cps(TY), "staged super-block as the host sizes it");
    constexpr int NW = 8, CPR = F::CPS | 1, NCH = 16 * F::CPS, NI = (NCH + 63) / 64;
    extern __shared__ uint4 smem[];
    const int nsb = a.cols >> 8, ns = (int)gridDim.y;
    int M = a.m, bx = blockIdx.x, gx = gridDim.x, pair0 = 0, slot = 0;
    if constexpr (GR) { /* gx blocks share a tile of up to T pairs of one slot */
        gx = a.ng;
        bool found;
        if (T == 16 && !(a.kw > 1 && gx == a.units)) { /* a share that the number of tiles can change */
            auto share = [&](int tiles) { return le_mtg_share(tiles, a.units, a.ng, a.kw, (int)gridDim.x, a.cus); };
            found = le_tile_shared(a.off, a.nslot, T, bx, share, gx, slot, pair0);
        } else {
            found = le_tile_of(a.off, a.nslot, T, bx / gx, slot, pair0);
        }
        if (!found) return; /* uniform: past the last tile */
        bx %= gx;
        M = min(T, a.off[slot + 1] - pair0);
    }
    const int sb0 = (int)blockIdx.y * nsb / ns, sb1 = ((int)blockIdx.y + 1) * nsb / ns, nsl = sb1 - sb0;
    const int most = (nsb + ns - 1) / ns; /* the launch's LDS holds the longest slice */
    uint4 *img = smem;
    float *stab = (float *)(smem + most * IMG);                /* [super-block][16 MFMA rows] */
    uint4 *stg = (uint4 *)(stab + most * 16);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = lane & 15;
    uint4 *wb = stg + wave * 16 * CPR;
    u8 *tab = (u8 *)(stg + NW * 16 * CPR);
    float4 *red = (float4 *)(tab + le_mt_tab(TY));              /* [2][NW][4 T lanes], with kw > 1 */
    if constexpr (le_mt_tab(TY) > 0) gq_tables<TY>(tab);

    const int KW = a.kw, RT = NW / KW, kw = wave % KW, rt = wave / KW;
    const int ntr = (a.rows + 15) >> 4, ntile = GR && a.dual ? 2 * ntr : ntr, mine = (nsl + KW - 1 - kw) / KW; /* super-blocks kw, kw + KW, ... of the slice */
    const size_t rb = (size_t)nsb * F::SBB;
    int ri[NI], gb[NI], wl[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int c = min(64 * i + lane, NCH - 1);
        ri[i] = c / F::CPS;
        gb[i] = F::goff(c % F::CPS);
        wl[i] = c + (CPR - F::CPS) * ri[i];
    }
    const u8 *w1 = a.w, *w2 = nullptr;
    if constexpr (GR) {
        w1 = a.ptrs ? a.ptrs[slot] : a.w + (size_t)slot * a.w_slot_bytes;
        if (a.dual) w2 = a.ptrs2 ? a.ptrs2[slot] : a.w2 + (size_t)slot * a.w_slot_bytes;
    }
    uint4 W[NI];
    auto issue = [&](int tile, int sb) {
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const u8 *p = (GR && tile >= ntr ? w2 : w1) + (size_t)min((GR && tile >= ntr ? tile - ntr : tile) * 16 + ri[i], a.rows - 1) * rb +
                          (size_t)sb * F::SBB + gb[i];
            W[i] = AL ? ldg16(p) : ldg16u(p);
        }
    };
    const int t0 = bx * RT, tstep = gx * RT;

    /* images: one (token, super-block) per wave and turn, four values per lane; a first batch of eight
     * turns' activations is loaded before the first weights (loads retire in order: behind them they
     * would wait for the weights) */
    {
        const int j = lane >> 3, g = (lane & 7) >> 1, np = M * nsl;
        const float inv = __builtin_amdgcn_rcpf((float)nsl);
        const LE_GLOBAL float4 *x4 = (const LE_GLOBAL float4 *)a.x;
        auto split = [&](int p, int &t, int &sl) { /* p = t nsl + sl; p < 2^12, and p + 1/2 keeps the quotient off the integers */
            t = __builtin_amdgcn_readfirstlane((int)(((float)p + 0.5f) * inv));
            sl = p - t * nsl;
        };
        float4 v[8];
        auto xload = [&](int p0) {
#pragma unroll
            for (int u = 0; u < 8; u++) {
                int t, sl;
                split(__builtin_amdgcn_readfirstlane(min(p0 + u * NW, np - 1)), t, sl);
                const size_t o = ((size_t)(GR ? a.in_idx[pair0 + t] : t) * a.cols + (size_t)(sb0 + sl) * 256) / 4 + lane;
                v[u] = x4[o];
                if (GR && a.up) v[u] = le_silu_mul4(v[u], ((const LE_GLOBAL float4 *)a.up)[o]);
            }
        };
        xload(wave);
        if (t0 + rt < ntile && mine > 0) issue(t0 + rt, sb0 + kw);
        for (int p0 = wave; p0 < np; p0 += 8 * NW) {
            if (p0 != wave) xload(p0);
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int p = __builtin_amdgcn_readfirstlane(p0 + u * NW);
                int t, sl;
                split(p, t, sl);
                if (p >= np) break; /* uniform over the wave */
                /* largest magnitude's exponent (the bits of a nonnegative float order as integers): 2^(ex + 9) <= max < 2^(ex + 10) */
                const float am = fmaxf(fmaxf(fabsf(v[u].x), fabsf(v[u].y)), fmaxf(fabsf(v[u].z), fabsf(v[u].w)));
                const int eb = mt_wave_max(__builtin_bit_cast(int, am)) >> 23, ex = eb == 0 || eb == 255 ? 0 : max(eb - 136, -100);
                const float sc = __builtin_bit_cast(float, (u32)(127 - ex) << 23), xv[4] = {v[u].x * sc, v[u].y * sc, v[u].z * sc, v[u].w * sc};
                _Float16 h[4], l[4];
                float hs = 0.f, ls = 0.f;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    h[i] = (_Float16)xv[i];
                    l[i] = (_Float16)((xv[i] - (float)h[i]) * 2048.f);
                    hs += (float)h[i];
                    ls += (float)l[i];
                }
                uint4 *ip = img + sl * IMG + (4 * j + g) * RS;
                ((uint2 *)(ip + t))[lane & 1] = make_uint2(as_u32((le_h2){h[0], h[2]}), as_u32((le_h2){h[1], h[3]}));
                if constexpr (HL) ((uint2 *)(ip + T + t))[lane & 1] = make_uint2(as_u32((le_h2){l[0], l[2]}), as_u32((le_h2){l[1], l[3]}));
                if constexpr (OFS) {
                    hs = mt_sum8(hs);
                    ls = mt_sum8(ls);
                    if ((lane & 7) == 0) { /* sub-block j at position P8(j), its sums' two halves in fragments 32 and 33 */
                        const int pj = (j & 4) | ((j & 1) << 1) | ((j >> 1) & 1);
                        uint4 *sp = img + sl * IMG + 32 * RS;
                        const _Float16 a0 = (_Float16)hs, b0 = (_Float16)ls;
                        ((_Float16 *)(sp + t))[pj] = a0;
                        ((_Float16 *)(sp + RS + t))[pj] = (_Float16)(hs - (float)a0);
                        if constexpr (HL) {
                            ((_Float16 *)(sp + T + t))[pj] = b0;
                            ((_Float16 *)(sp + RS + T + t))[pj] = (_Float16)(ls - (float)b0);
                        }
                    }
                }
                if (lane == 0) {
                    stab[sl * 16 + t] = __builtin_bit_cast(float, (u32)(127 + ex) << 23);
                    if constexpr (HL) stab[sl * 16 + T + t] = __builtin_bit_cast(float, (u32)(116 + ex) << 23);
                }
            }
        }
    }
    __syncthreads();

    float *out1 = a.part ? a.part + (size_t)blockIdx.y * a.m * a.rows : a.y;
    int par = 0;
    for (int tb = t0; tb < ntile; tb += tstep) {
        const int tile = tb + rt;
        le_v4f y = {0.f, 0.f, 0.f, 0.f};
        if (tile < ntile) {
            for (int i = 0; i < mine; i++) {
                const int sl = kw + i * KW;
#pragma unroll
                for (int u = 0; u < NI; u++) wb[wl[u]] = W[u];
                int nt = tile, nsl_ = sl + KW;
                if (nsl_ >= nsl) { nsl_ = kw; nt += tstep; }
                if (nt < ntile) issue(nt, sb0 + nsl_);
                mt_sb<TY, R, RS>((const u8 *)(wb + n * CPR), img + sl * IMG, lane, *(const float4 *)(stab + sl * 16 + 4 * (lane >> 4)), tab, y);
            }
        }
        /* high and low halves of a token lie T rows apart: lanes 4 T apart */
        if constexpr (HL) {
#pragma unroll
            for (int e = 0; e < 4; e++) y[e] += __shfl_xor(y[e], 4 * T);
        }
        if (KW > 1) {
            float4 *rp = red + par * NW * 4 * T;
            if (lane < 4 * T) rp[wave * 4 * T + lane] = make_float4(y[0], y[1], y[2], y[3]);
            __syncthreads();
            if (kw == 0 && lane < 4 * T)
                for (int k = 1; k < KW; k++) {
                    const float4 v = rp[(wave + k) * 4 * T + lane];
                    y[0] += v.x;
                    y[1] += v.y;
                    y[2] += v.z;
                    y[3] += v.w;
                }
            par ^= 1;
        }
        const bool second = GR && tile >= ntr;
        float *out = second ? a.y2 : out1;
        const int r = (second ? tile - ntr : tile) * 16 + n;
        if (kw == 0 && lane < 4 * T && tile < ntile && r < a.rows) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int t = 4 * (lane >> 4) + e;
                if (t < M) out[(size_t)(GR ? a.out_idx[pair0 + t] : t) * a.rows + r] = y[e];
            }
        }
    }
}

#define LE_MT_(TY, T) \
    extern "C" __global__ void __launch_bounds__(512) le_mt_##TY##_t##T(MtArgs a) { mt_body<TY, T, T <= 8, false>(a); }
#define LE_MTG_(TY, T) \
    extern "C" __global__ void __launch_bounds__(512) le_mtg_##TY##_t##T(MtArgs a) { mt_body<TY, T, false, true>(a); }
#define LE_MT(TY) LE_MT_(TY, 4) LE_MT_(TY, 8) LE_MT_(TY, 16) LE_MTG_(TY, 8) LE_MTG_(TY, 16)
LE_MT(2) LE_MT(8) LE_MT(11) LE_MT(12) LE_MT(13) LE_MT(14) LE_MT(16) LE_MT(18) LE_MT(22)
