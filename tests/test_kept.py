"""The tables that a handle keeps by key (kept.h), compiled for the CPU: what
cannot be built is tried once, the least recently used goes first, and what a
sweep adds is gone afterwards and nothing else."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cstdio>
#include <cstdlib>
#include <set>
#include "kept.h"

static int tries = 0;
static bool can = true;
static std::set<int> live;  // values made and not dropped

#define CHECK(x) \
  do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); std::exit(1); } } while (0)

int main() {
  tt::Kept<int, int> k(3);
  auto drop = [](int v) { CHECK(live.erase(v) == 1); };
  auto get = [&](int key, bool build, bool again = false) {
    return k.get(key, build, again, [&](int* v) {
      ++tries;
      if (can) live.insert(*v = 100 + key);
      return can;
    }, drop);
  };
  // a failure is not tried again, but on request
  can = false;
  for (int i = 0; i < 5; ++i) CHECK(!get(1, true));
  CHECK(tries == 1);
  CHECK(!get(1, true, true) && tries == 2);
  can = true;
  CHECK(!get(1, true) && tries == 2);
  CHECK(*get(1, true, true) == 101 && tries == 3);
  CHECK(*get(1, true) == 101 && *get(1, false) == 101 && tries == 3);
  // nothing is built without leave
  CHECK(!get(2, false) && tries == 3);
  // the least recently used goes
  CHECK(get(2, true) && get(3, true) && get(1, false) && get(4, true));
  CHECK(k.size() == 3 && !get(2, false) && get(1, false) && get(3, false) && get(4, false));
  CHECK(live == (std::set<int>{101, 103, 104}));
  // a sweep: one at a time beyond the three, none of them left, none of before lost
  for (int key = 10; key < 20; ++key) {
    const auto m = k.mark();
    can = key != 12;
    CHECK(!get(key, true) == (key == 12));
    k.back_to(m, drop);
    CHECK(live == (std::set<int>{101, 103, 104}));
  }
  can = true;
  tries = 0;
  CHECK(get(12, true) && tries == 1);  // its failure is forgotten too
  // failures are bounded
  can = false;
  for (int key = 1000; key < 2000; ++key) CHECK(!get(key, true));
  k.clear(drop);
  CHECK(live.empty() && k.size() == 0);
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")
def test_kept_tables(tmp_path):
    src = tmp_path / "kept_checks.cpp"
    src.write_text(SOURCE)
    exe = str(tmp_path / "kept_checks")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined",
                    "-I", os.path.join(ROOT, "tentaco_amd", "csrc"), str(src), "-o", exe],
                   check=True, timeout=120)
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
