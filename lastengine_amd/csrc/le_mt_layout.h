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

/* Grouped form. The most tiles of T pairs that any routing of npair pairs to nslot slots makes. */
constexpr int le_mtg_tiles(int npair, int nslot, int T) {
    const int live = npair < nslot ? npair : nslot;
    return live + (npair - live) / T;
}
/* Blocks of a launch over at most `tiles` tiles, each of `units` groups of row tiles, that an even routing shares
 * between ng blocks. With 16 pairs a tile, and more tiles than half of the `cus` CUs, there is room for two rounds of
 * blocks: an uneven routing may then be dealt in smaller pieces (blocks without work cost 0.5 us of a small launch). */
constexpr int le_mtg_grid(int tiles, int units, int T, int ng, int cus) {
    const long long all = (long long)tiles * units, even = (long long)tiles * ng, two = T == 16 && 2 * tiles > cus ? 2LL * cus : 0;
    return (int)(even > two ? even : all < two ? all : two);
}
/* 16 pairs a tile: blocks that share each of `tiles` tiles in that launch (kw waves a row tile). The host does not see
 * the routing: only the device knows the number of tiles, a third of the even routing's where all tokens take the same
 * experts. The even routing's share where its blocks fill more than half of the CUs once, or cannot be cut further;
 * else the share whose rounds of blocks (their images leave room for little more than one a CU) are the shortest, the
 * images of a tile counted as one and a half groups. 128 experts, 8 a token, 48 / 64 / 96 tokens to the same eight, the
 * fixed share against this: 768 x 2048 Q4_K 36.6 / 37.2 / 37.1 -> 22.0 / 22.5 / 31.2 us, 2048 x 768 39.2 / 39.9 / 40.2 ->
 * 16.8 / 16.9 / 25.2; half of 96 tokens' pairs to eight 61.0 -> 52.1 (Q6_K 84.2 -> 68.4); an even routing within 3%. */
constexpr int le_mtg_share(int tiles, int units, int ng, int kw, int grid, int cus) {
    if (tiles * ng > cus ? kw > 1 : 2 * tiles * ng > cus || ng == units) return ng;
    int cost = 0x7FFFFFFF;
    for (int per = 1; per <= 8; per++) { /* groups a block takes */
        const int n = (units + per - 1) / per, nb = tiles * n;
        const int c = (nb + cus - 1) / cus * (2 * per + 3);
        if (nb <= grid && c < cost) {
            cost = c;
            ng = n;
        }
    }
    return ng;
}
