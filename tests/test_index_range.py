"""The kernels' index arithmetic at the top of the int32 range of a CSF (2^30
level N-2 nodes and more, 2^31 - 1 nonzeros), where sums of two int32 values
pass it: the functions they use, compiled for the CPU with integer overflow
trapped. (Tensors of that size do not fit a test; the kernels themselves run in
the GPU tests of the level modes and the edge walk.)"""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <climits>
#include <cstdio>
#include <cstdlib>
#include "index_range.h"

static void expect(long long got, long long want, const char* what) {
  if (got == want) return;
  std::printf("%s: %lld, not %lld\n", what, got, want);
  std::exit(1);
}

int main() {
  using namespace tt;
  // the first entry whose end lies past int32, and the last there can be
  expect(index_end(1 << 30, (1 << 30) - 1), (1ll << 31) - 1, "end below");
  expect(index_end(1 << 30, 1 << 30), 1ll << 31, "end at");
  expect(index_end(INT_MAX, INT_MAX - 1), 2ll * INT_MAX - 1, "end of the last");
  expect(index_end(3, 2), 5, "end of a few");
  for (int lane = 0; lane <= 64; ++lane) {
    expect(index_ahead(INT_MAX - 1, lane, INT_MAX - 1), INT_MAX - 1, "from the last");
    expect(index_ahead(INT_MAX - 40, lane, INT_MAX - 1), lane < 39 ? INT_MAX - 40 + lane : INT_MAX - 1, "across");
    expect(index_ahead(0, lane, 0), 0, "one");
    expect(index_ahead(5, lane, 37), lane < 32 ? 5 + lane : 37, "inside");
  }
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")
def test_index_arithmetic_at_the_top_of_the_range(tmp_path):
    src = tmp_path / "index_checks.cpp"
    src.write_text(SOURCE)
    exe = str(tmp_path / "index_checks")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize-recover=undefined",
                    "-I", os.path.join(ROOT, "tentaco_amd", "csrc"), str(src), "-o", exe],
                   check=True, timeout=120)
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
