"""CPU check of the bookkeeping behind megakernel_reset (csrc/mk_written.h):
rows count as zero only once their clear was issued."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include <vector>
#include "mk_written.h"
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
  mk::WrittenRows w;
  std::vector<long long> asked;
  bool works = true;
  const auto clear = [&](long long rows) { asked.push_back(rows); return works; };
  CHECK(w.clear(clear) && asked.empty());  // nothing written: nothing to clear
  w.wrote(33), w.wrote(7);
  works = false;
  CHECK(!w.clear(clear) && asked.back() == 64);  // could not be issued
  w.wrote(5);
  works = true;
  CHECK(w.clear(clear) && asked.back() == 64);  // the next one covers the same rows
  const size_t n = asked.size();
  CHECK(w.clear(clear) && asked.size() == n);
  w.wrote(32);
  CHECK(w.clear(clear) && asked.back() == 32);
  w.wrote(0x7fffffff);
  CHECK(w.clear(clear) && asked.back() == 0x80000000LL);
  std::puts("ok");
}
"""


def test_rows_stay_written_until_their_clear_was_issued(tmp_path):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    src, out = tmp_path / "written.cpp", tmp_path / "written"
    src.write_text(SRC)
    subprocess.run([gxx, "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "megakernel_amd", "csrc"),
                    str(src), "-o", str(out)], check=True, timeout=120)
    r = subprocess.run([str(out)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout
