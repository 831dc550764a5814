/* Shared by the matrix-core GEMM kernels: the grouped form's tiles, conversions of packed codes to halves and the IQ
 * lookup tables in fragment order (the eight K positions of a lane's fragment in the order P8 = 0,2,1,3,4,6,5,7,
 * what the byte-pair conversion produces). */
#pragma once
#include "le_qmm_device.h"
#include "le_iq_tables.h"

typedef _Float16 le_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 le_v8h __attribute__((ext_vector_type(8)));
typedef float le_v16f __attribute__((ext_vector_type(16)));

__device__ const u32 le_gq_iq2_grid[512] = LE_IQ2XXS_GRID_WORDS;
__device__ const u32 le_gq_iq3_grid[256] = LE_IQ3XXS_GRID_WORDS;
__device__ const u32 le_gq_iq2s_grid[2048] = LE_IQ2S_GRID_WORDS;

__device__ __forceinline__ le_h2 as_h2(u32 v) { return __builtin_bit_cast(le_h2, v); }
__device__ __forceinline__ u32 as_u32(le_h2 v) { return __builtin_bit_cast(u32, v); }
__device__ __forceinline__ le_v8h as_v8h(uint4 v) { return __builtin_bit_cast(le_v8h, v); }

/* bytes 0 and 2 (lo) or 1 and 3 (hi) of w, each under the fp16 exponent of 1024 */
__device__ __forceinline__ u32 h1024_02(u32 w) { return __builtin_amdgcn_perm(0x64646464u, w, 0x04020400u); }
__device__ __forceinline__ u32 h1024_13(u32 w) { return __builtin_amdgcn_perm(0x64646464u, w, 0x04030401u); }
/* byte i of w duplicated into both halves under the exponent of 1024 */
__device__ __forceinline__ u32 h1024_dup(u32 w, int i) {
    const u32 sel = 0x04000400u | (u32)(i * 0x00010001);
    return __builtin_amdgcn_perm(0x64646464u, w, sel);
}
/* (x & m) | c in one instruction: the compiler otherwise emits an and and an or, because a VOP3
 * instruction cannot carry the two literal constants; m and c stay in registers */
__device__ __forceinline__ u32 and_or(u32 x, u32 m, u32 c) {
    u32 r;
    __asm__("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(m), "v"(c));
    return r;
}
__device__ __forceinline__ u32 pk_fma(u32 a, u32 b, u32 c) {
    return as_u32(__builtin_elementwise_fma(as_h2(a), as_h2(b), as_h2(c)));
}
__device__ __forceinline__ u32 pk_add(u32 a, u32 b) { return as_u32(as_h2(a) + as_h2(b)); }
__device__ __forceinline__ u32 pk_mul(u32 a, u32 b) { return as_u32(as_h2(a) * as_h2(b)); }
__device__ __forceinline__ u32 h2dup(float f) {
    const _Float16 h = (_Float16)f;
    return as_u32((le_h2){h, h});
}

/* IQ tables in LDS, in fragment order: grid entries as fp16 magnitudes (IQ2_XXS, IQ2_S: 8 per
 * entry, P8 order; IQ3_XXS: 4 per entry, order 0,2,1,3), then for each 7-bit sign index the 8 half
 * masks of ksign (src/quant.rs:57), or for IQ2_S for each sign byte its 8 bits (src/quant.rs:155-167),
 * 0x8000 where the value is negative, P8 order. */
template <int TY>
__device__ __forceinline__ void gq_tables(u8 *tab) {
    if constexpr (TY == LE_TYPE_IQ2_XXS || TY == LE_TYPE_IQ3_XXS || TY == LE_TYPE_IQ2_S) {
        constexpr int NG = TY == LE_TYPE_IQ2_S ? 1024 : 256, GB = TY == LE_TYPE_IQ3_XXS ? 8 : 16;
        for (int i = threadIdx.x; i < NG; i += blockDim.x) {
            if constexpr (TY != LE_TYPE_IQ3_XXS) {
                const u32 *gw = TY == LE_TYPE_IQ2_S ? le_gq_iq2s_grid : le_gq_iq2_grid;
                const u32 w0 = gw[2 * i], w1 = gw[2 * i + 1];
                *(uint4 *)(tab + GB * i) = make_uint4(pk_add(h1024_02(w0), 0xE400E400u), pk_add(h1024_13(w0), 0xE400E400u),
                                                      pk_add(h1024_02(w1), 0xE400E400u), pk_add(h1024_13(w1), 0xE400E400u));
            } else {
                const u32 w0 = le_gq_iq3_grid[i];
                *(uint2 *)(tab + GB * i) = make_uint2(pk_add(h1024_02(w0), 0xE400E400u), pk_add(h1024_13(w0), 0xE400E400u));
            }
        }
        /* IQ2_S stores its 8 sign bits explicitly: 256 entries indexed by the sign byte */
        constexpr int NS = TY == LE_TYPE_IQ2_S ? 256 : 128;
        u8 *sg = tab + NG * GB;
        for (int i = threadIdx.x; i < NS; i += blockDim.x) {
            const u32 ks = NS == 256 ? (u32)i : (u32)i | ((__builtin_popcount((u32)i) & 1u) << 7);
            u32 m[4];
#pragma unroll
            for (int p = 0; p < 4; p++) { /* halves 2p, 2p+1 hold values P8(2p), P8(2p+1) */
                const int v0 = (p & 2) * 2 + (p & 1), v1 = v0 + 2;
                m[p] = (((ks >> v0) & 1u) << 15) | (((ks >> v1) & 1u) << 31);
            }
            *(uint4 *)(sg + 16 * i) = make_uint4(m[0], m[1], m[2], m[3]);
        }
    }
}

/* Tiles of the grouped form: slot s has off[s+1] - off[s] pairs, split into tiles of bm, listed
 * slot by slot. Each wave derives what it needs from off itself (no planning launch): the slots'
 * counts are loaded 256 at a time, all in flight together, then scanned across the wave. */
__device__ __forceinline__ int le_wave_scan(int v) { /* inclusive prefix sum over the wave, by DPP */
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true); /* row_shr:1 (rows of 16 lanes) */
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true); /* row_shr:2 */
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true); /* row_shr:4 */
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true); /* row_shr:8 */
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false); /* row_bcast:15 into rows 1, 3 */
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false); /* row_bcast:31 into rows 2, 3 */
    return v;
}
/* Walk the slots 256 at a time (every load of a round in flight together), each lane holding one
 * slot's first pair o0, its tile count c and the number of tiles before it; stop at the first
 * slot for which hit(o0, o1, first, c) holds on some lane. Returns that slot (or -1) and, through
 * the references, its first pair and first tile. Uniform over the wave. */
template <class Hit>
__device__ __forceinline__ int le_slot_walk(const int *__restrict__ off, int nslot, int bm, Hit hit, int &o0_out, int &first_out) {
    const int lane = threadIdx.x & 63;
    int base = 0;
    for (int s0 = 0; s0 < nslot; s0 += 256) {
        int o0[4], o1[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int s = min(s0 + 64 * q + lane, nslot - 1);
            o0[q] = off[s];
            o1[q] = off[s + 1];
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const bool in = s0 + 64 * q + lane < nslot;
            const int c = in ? (max(o1[q] - o0[q], 0) + bm - 1) / bm : 0, inc = le_wave_scan(c), first = base + inc - c;
            const unsigned long long h = __ballot(in && c > 0 && hit(o0[q], o1[q], first, c));
            if (h) {
                const int l = __ffsll((long long)h) - 1;
                o0_out = __shfl(o0[q], l);
                first_out = __shfl(first, l);
                return s0 + 64 * q + l;
            }
            base += __shfl(inc, 63);
        }
    }
    return -1;
}
/* A round of the walk: 256 slots from s0, every load in flight together; lane l of group q holds slot s0 + 64 q + l's
 * pairs o0 .. o1, its tile count c and the number of tiles before it, first (from base tiles of earlier rounds). */
struct LeRound {
    int o0[4], o1[4], c[4], first[4];
};
__device__ __forceinline__ LeRound le_slot_round(const int *__restrict__ off, int nslot, int bm, int s0, int &base) {
    const int lane = threadIdx.x & 63;
    LeRound r;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if (s0 + 64 * q >= nslot) break; /* uniform */
        const int s = min(s0 + 64 * q + lane, nslot - 1);
        r.o0[q] = off[s];
        r.o1[q] = off[s + 1];
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        r.c[q] = 0;
        if (s0 + 64 * q >= nslot) continue; /* uniform */
        if (s0 + 64 * q + lane < nslot) r.c[q] = (max(r.o1[q] - r.o0[q], 0) + bm - 1) / bm;
        const int inc = le_wave_scan(r.c[q]);
        r.first[q] = base + inc - r.c[q];
        base += __builtin_amdgcn_readlane(inc, 63);
    }
    return r;
}
/* tile mt: its slot and first pair (false past the last tile) */
__device__ __forceinline__ bool le_tile_of(const int *__restrict__ off, int nslot, int bm, int mt, int &slot, int &pair0) {
    int o0, first;
    slot = le_slot_walk(off, nslot, bm, [mt](int, int, int f, int c) { return mt >= f && mt < f + c; }, o0, first);
    pair0 = o0 + (mt - first) * bm;
    return slot >= 0;
}
/* Block bx of a launch whose blocks share the tiles, share(tiles) blocks each (most often the given ng): that number, the
 * tile's slot and its first pair (false past the last tile). The first round's offsets serve the count and the search. */
template <class Share>
__device__ __forceinline__ bool le_tile_shared(const int *__restrict__ off, int nslot, int bm, int bx, Share share, int &ng, int &slot, int &pair0) {
    int base = 0, mt = bx / ng; /* the division while the offsets load */
    const LeRound r = le_slot_round(off, nslot, bm, 0, base);
    const int in0 = base, even = ng;
    for (int s0 = 256; s0 < nslot; s0 += 256) le_slot_round(off, nslot, bm, s0, base);
    ng = share(base);
    if (ng != even) mt = bx / ng;
    if (mt >= base) return false;
    if (mt >= in0) return le_tile_of(off, nslot, bm, mt, slot, pair0);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if (64 * q >= nslot) break; /* uniform */
        const unsigned long long h = __ballot(r.c[q] && mt >= r.first[q] && mt < r.first[q] + r.c[q]);
        if (h) {
            const int l = __ffsll((long long)h) - 1;
            slot = 64 * q + l;
            pair0 = __builtin_amdgcn_readlane(r.o0[q], l) + (mt - __builtin_amdgcn_readlane(r.first[q], l)) * bm;
        }
    }
    return true;
}
