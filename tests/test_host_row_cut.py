"""The cut of a long row into segments (cut_long_row of grd_internal.hpp), built
with g++: whole, in order, none longer than asked for, and with an end for rows
up to the largest arc count a graph may have, 2^32 - 17 (no GPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "grd_internal.hpp"
int main(int, char **argv)
{
  const uint32_t e0 = strtoul(argv[1], 0, 0), e1 = strtoul(argv[2], 0, 0), n = strtoul(argv[3], 0, 0);
  uint64_t at = e0, k = 0;
  const uint32_t nseg = grd::cut_long_row(e0, e1, n, [&](uint32_t a, uint32_t b) {
    if (a != at || b <= a || b - a > n || b > e1 || ++k > (1u << 24)) {
      std::printf("wrong segment %u %u\n", a, b);
      exit(1);
    }
    at = b;
  });
  if (at != e1 || nseg != k || nseg != ((uint64_t)e1 - e0 + n - 1) / n) return 2;
  return 0;
}
"""


@pytest.fixture(scope="module")
def cut(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None or not os.path.exists(os.path.join(ROCM, "include", "hip", "hip_runtime.h")):
        pytest.skip("no g++ or HIP headers on this machine")
    d = tmp_path_factory.mktemp("cut")
    src, exe = d / "cut.cpp", d / "cut"
    src.write_text(PROGRAM)
    subprocess.run([gxx, "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROCM, "include"),
                    "-I", os.path.join(ROOT, "grudon_amd", "csrc"), "-I", os.path.join(ROOT, "include"), str(src),
                    "-o", str(exe)], check=True)
    return str(exe)


@pytest.mark.parametrize("n", [504, 2048, 4096, 16384])
@pytest.mark.parametrize("e0,length", [(0, 1), (5, 504), (5, 16385), (0, 2 ** 32 - 17), (7, 2 ** 32 - 24),
                                       (2 ** 32 - 17 - 40000, 40000), (2 ** 32 - 17 - 16385, 16385)])
def test_segments(cut, n, e0, length):
    p = subprocess.run([cut, str(e0), str(e0 + length), str(n)], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0, p.stdout
