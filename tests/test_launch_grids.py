"""Launch grids (mb_grid.h) below the 2^32 threads of a dimension."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include <initializer_list>
#include "mb_grid.h"
using mb::launch_blocks;
int main() {
    for (int threads : {64, 256, 512, 1024})
        for (int64_t want = 0; want < ((int64_t)1 << 33); want = want < 16 ? want + 1 : want * 2 + 1) {
            const int64_t b = launch_blocks(want, threads);
            if (b < 1 || b * threads >= (int64_t)1 << 32) return 1;
            if (want >= 1 && want * threads < (int64_t)1 << 32 && b != want) return 2;
        }
    return launch_blocks(8388607, 512) == 8388607 && launch_blocks(8388608, 512) == 8388607 ? 0 : 3;
}
"""


def test_blocks(tmp_path):
    (tmp_path / "p.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", f"-I{ROOT / 'mojoboost_amd' / 'csrc'}", str(tmp_path / "p.cpp"), "-o",
                    str(tmp_path / "p")], check=True)
    assert subprocess.run([str(tmp_path / "p")]).returncode == 0
