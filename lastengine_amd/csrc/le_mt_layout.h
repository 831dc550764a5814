/* What the few-token kernels (le_mt_*, le_mtg_*) and the host that launches them share: the LDS of a block
 * and the staged super-blocks it holds. Plain C++17: the host, the device pass and a CPU test include it. */
#pragma once
#include <cstddef>

/* 16-byte chunks of a staged super-block */
constexpr int le_mt_cps(int ty) {
    return ty == 14 /* Q6_K */ ? 14 : ty == 16 /* IQ2_XXS */ ? 5 : ty == 18 /* IQ3_XXS */ ? 7 : ty == 8 /* Q8_0 */ ? 17
         : ty == 13 /* Q5_K */ ? 11 : ty == 11 /* Q3_K */ ? 7 : ty == 22 /* IQ2_S */ ? 6 : 9 /* Q4_K, Q4_0 */;
}
/* bytes of the IQ lookup tables */
constexpr int le_mt_tab(int ty) { return ty == 16 ? 6144 : ty == 18 ? 4096 : ty == 22 ? 20480 : 0; }

/* A block of 8 waves: images of `most` super-blocks with R live MFMA rows (fragments of R + 1 slots, two more for
 * the offset sums of Q4_K and Q5_K) and their scales, each wave's 16 staged rows, tables, the waves' sums
 * for T tokens (two buffers, where several waves share a row tile). */
constexpr size_t le_mt_lds(int ty, int most, int R, int T, bool sums) {
    return (size_t)most * ((size_t)(ty == 12 || ty == 13 ? 34 : 32) * (R + 1) * 16 + 64) + (size_t)8 * 16 * (le_mt_cps(ty) | 1) * 16 +
           le_mt_tab(ty) + (sums ? (size_t)2 * 8 * 4 * T * 16 : 0);
}

/* Q8_0, Q4_0: the 8 values' bytes of group g (Q4_0: of nibble pairs, g of 0, 1) of sub-block j start at byte
 * le_mt_byte of the staged super-block, 4-byte aligned where j is odd, else 2-byte aligned: that many words are read. */
constexpr int le_mt_byte(int ty, int j, int g) { return (ty == 8 ? 34 : 18) * j + 2 + 8 * g; }
constexpr int le_mt_words(int j) { return j & 1 ? 2 : 3; }
