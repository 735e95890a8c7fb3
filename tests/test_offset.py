"""The 32-bit x offsets of vnec_spmm.hip (vnec_offset.h) on the CPU, compiled
so that signed overflow traps: rows around and beyond 2 GiB of x, up to the
4 GiB from which the kernels take 64-bit offsets."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = """
#include <stdlib.h>
#include "vnec_offset.h"
int main(int argc, char **argv)
{
    const int64_t x_bytes = strtoll(argv[1], 0, 0);
    const int k = atoi(argv[2]), lanes = k < 8 ? k / 2 : 4, part = 8 * k / lanes;
    volatile int32_t row = (int32_t)(x_bytes / (8 * k) - 1);
    for (volatile int32_t q = 0; q < lanes; q++)
        if (vnec_x_offset(row, 8 * k, q, part) != (uint64_t)row * 8 * k + (uint64_t)q * part) return 1;
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("offset")
    (d / "offset.c").write_text(PROGRAM)
    exe = str(d / "offset")
    subprocess.run(["gcc", "-O0", "-ftrapv", "-I", os.path.join(ROOT, "vnec_amd", "csrc", "hip"),
                    str(d / "offset.c"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("k", [2, 4, 8, 16])
@pytest.mark.parametrize("x_bytes", [1 << 20, 1 << 31, (1 << 31) + 128, 3 << 30, (1 << 32) - 128])
def test_x_offsets_to_4_gib(program, x_bytes, k):
    assert subprocess.run([program, str(x_bytes), str(k)]).returncode == 0
