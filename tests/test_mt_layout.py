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
