"""Every byte that the 256-row expert tile loads of an expert's matrix (csrc/hybrid/moe_tile.h, the kernel's own address arithmetic) lies inside
it, in the last tile of a matrix that ends with half of one too, and rows that exist are loaded from where they are."""
import os
import shutil
import subprocess

import pytest

WALK = r"""
#include "moe_tile.h"
#include <cstdio>
#include <cstdlib>
int main(int argc, char** argv) {
    const int N = atoi(argv[1]), K = atoi(argv[2]);
    const int64_t bytes = (int64_t)N * K * 2;
    for (int tn = 0; tn < (N + 255) / 256; ++tn)
        for (int wave = 0; wave < 8; ++wave)
            for (int i = 0; i < 4; ++i)
                for (int lane = 0; lane < 64; ++lane) {
                    const int64_t at = chronos::hy::moe_weight_offset(tn, wave, i, lane, N, K);
                    if (at < 0 || at + (K / 64 - 1) * 128 + 16 > bytes) return 1;
                    const int row = tn * 256 + 32 * wave + 8 * i + lane / 8;
                    if (row < N && at != (int64_t)row * K * 2 + ((lane & 7) ^ (row & 7)) * 16) return 2;
                }
    puts("inside");
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("moe_tile")
    (d / "walk.cpp").write_text(WALK)
    inc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "csrc", "hybrid")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I" + inc, str(d / "walk.cpp"), "-o", str(d / "walk")], check=True)
    return str(d / "walk")


@pytest.mark.parametrize("N,K", [(128, 128), (256, 128), (384, 512), (1408, 2048), (11 * 128, 4096), (2048, 1408), (8191 * 128, 1024)])
def test_inside(walk, N, K):
    assert N * K * 2 < 1 << 31
    out = subprocess.run([walk, str(N), str(K)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout == "inside\n"
