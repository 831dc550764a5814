"""Host-side checks of the few-token kernels' LDS layout (lastengine_amd/csrc/le_mt_layout.h), which the kernels
and the host that sizes their launches share."""
import os
import subprocess

from tests.conftest import REPO

PROG = r"""
#include <cstdio>
#include <initializer_list>
#include "le_mt_layout.h"
int main() {
    for (int ty : {8, 2})
        for (int j = 0; j < 8; j++)
            for (int g = 0; g < (ty == 8 ? 4 : 2); g++)
                std::printf("%d %d %d %d %d %d\n", ty, j, g, le_mt_byte(ty, j, g), le_mt_words(j), 16 * le_mt_cps(ty));
}
"""


def test_staged_reads_stay_inside_the_super_block(tmp_path):
    """Q8_0 and Q4_0: the words read for a group of 8 values hold its bytes and end with the staged super-block: the
    last row of a block's last wave ends its LDS where one wave takes a row tile (no sums behind it)."""
    src, exe = tmp_path / "layout.cpp", str(tmp_path / "layout")
    src.write_text(PROG)
    subprocess.run(["g++", "-std=c++17", "-I" + os.path.join(REPO, "lastengine_amd", "csrc"), str(src), "-o", exe], check=True)
    lines = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.splitlines()
    assert len(lines) == 8 * 4 + 8 * 2
    for line in lines:
        ty, j, g, byte, words, size = map(int, line.split())
        assert byte == (34 if ty == 8 else 18) * j + 2 + 8 * g
        first, last = byte & ~3, (byte & ~3) + 4 * words
        assert first <= byte and byte + 8 <= last <= size, (ty, j, g)


SHARE = r"""
#include <cstdio>
#include "le_mt_layout.h"
int main() {
    int npair, nslot, units, T, ng, tiles;
    while (std::scanf("%d %d %d %d %d %d", &npair, &nslot, &units, &T, &ng, &tiles) == 6) {
        const int most = le_mtg_tiles(npair, nslot, T), grid = le_mtg_grid(most, units, T, ng, 256);
        std::printf("%d %d %d\n", most, grid, T == 16 ? le_mtg_share(tiles, units, ng, 1, grid, 256) : ng);
    }
}
"""


def test_grouped_blocks_cover_any_routing(tmp_path):
    """Few-pair grouped form: whatever the routing, its tiles are at most those the host counts on and the grid holds
    the blocks that share them; a routing of every token to the same experts is dealt to more of the chip."""
    import numpy as np
    src, exe = tmp_path / "share.cpp", str(tmp_path / "share")
    src.write_text(SHARE)
    subprocess.run(["g++", "-std=c++17", "-I" + os.path.join(REPO, "lastengine_amd", "csrc"), str(src), "-o", exe], check=True)

    def run(cases):
        out = subprocess.run([exe], input="\n".join(" ".join(map(str, c)) for c in cases), check=True, capture_output=True, text=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    rng = np.random.default_rng(0)
    cases = []
    for nslot in (1, 2, 7, 32, 128, 300):
        for npair in sorted({1, 2, nslot, 2 * nslot, 2 * nslot + 1, 4 * nslot, 6 * nslot}):
            T = 8 if npair <= 2 * nslot else 16
            for hot in (1, min(8, nslot), nslot):
                counts = rng.multinomial(npair, np.ones(hot) / hot)
                ragged = np.full(nslot, 0)  # one pair past a tile in as many slots as there can be
                ragged[:min(nslot, npair // (T + 1))] = T + 1
                ragged[-1] += npair - ragged.sum()
                for c in (counts, ragged):
                    for units, per in ((1, 1), (6, 2), (12, 6), (16, 8), (128, 8), (128, 3)):
                        cases.append((npair, nslot, units, T, -(-units // per), int(np.sum(-(-c // T)))))
    rows = run(cases)
    assert len(rows) == len(cases)
    for case, (most, grid, share) in zip(cases, rows):
        tiles, units = case[5], case[2]
        assert tiles <= most and 1 <= share <= units and tiles * share <= grid, (case, most, grid, share)
    # 512 pairs of 128 experts, 12 groups of row tiles shared by two blocks under an even routing: 126 tiles of one, and
    # the 32 tiles of a routing to eight experts, spread over more than the 64 blocks of that share
    (_, _, even), (_, _, hot) = run([(512, 128, 12, 16, 2, 126), (512, 128, 12, 16, 2, 32)])
    assert even == 2 and 32 * hot > 128
