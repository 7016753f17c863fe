"""The block of 1 x 3 x 3 base voxels that a sampling point is filed under (csrc/d2c_brick.hpp): every base voxel that the axes of the sorted points
can have (they end below 2^23) against division by repeated counting, on the host."""
import os
import subprocess

from d2conv3d_amd import build

PROGRAM = r"""
#include <cstdio>
#include "d2c_brick.hpp"
int main()
{
    int block = 0, in = 0;                       // of base voxel -1
    for (int v = -1; v < (1 << 23); v++) {
        if (brick_block(v) != block) { std::printf("base voxel %d: block %d, not %d\n", v, brick_block(v), block); return 1; }
        if (++in == 3) { in = 0; block++; }
    }
    return 0;
}
"""


def test_block_of_every_base_voxel(tmp_path):
    src, exe = tmp_path / "blocks.hip", tmp_path / "blocks"
    src.write_text(PROGRAM)
    subprocess.run([build.HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-O2", "-std=c++17", f"-I{build.CSRC}", str(src), "-o", str(exe)],
                   check=True, capture_output=True, text=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
