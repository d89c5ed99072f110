"""The sparse MLA's page-table reads (csrc/mla_table.h, the kernels' own code, built here
for the CPU, with every read kept): a row's request id is followed only for a position in
use.  The table lies between two pages that may not be touched, so a read outside it ends
the program."""

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "sgl-amd-mono_amd" / "csrc"

MAIN = r"""
#include <stdio.h>
#include <sys/mman.h>
#include <initializer_list>
#include "mla_table.h"
int main() {
  const size_t P = 4096;
  char* m = (char*)mmap(nullptr, 3 * P, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0);
  if (m == MAP_FAILED || mprotect(m + P, P, PROT_READ | PROT_WRITE)) return 2;
  int32_t* pt = (int32_t*)(m + P);  // [4][256]
  const int stride = 256;
  for (int i = 0; i < 1024; ++i) pt[i] = 5000 + i;
  // requests 0 and 3 decode; rows 2 .. 5 are pad rows whose request id says nothing
  const int32_t req[] = {0, 3, -1, 4, 1 << 30, INT32_MIN};
  for (int r = 0; r < 6; ++r)
    for (int pos : {-1, 0, 63, 64, 16383, 16384, INT32_MAX, INT32_MIN}) {
      const bool used = pos >= 0 && pos < stride * 64;
      if (r >= 2 && used) continue;
      const int row = mk2::mla_cache_row(pos, mk2::mla_page(pt, mk2::mla_line(req, r, stride), stride, pos), stride);
      const int want = used ? (5000 + req[r] * stride + pos / 64) * 64 + pos % 64 : -1;
      if (row != want) return printf("row %d pos %d: %d, not %d\n", r, pos, row, want), 1;
    }
  puts("ok");
}
"""


def test_unused_entries_leave_the_page_table_alone(tmp_path):
    cxx = shutil.which("g++") or pytest.skip("no host compiler")
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "main"
    subprocess.run([cxx, "-std=c++17", "-O0", "-I", str(CSRC), str(tmp_path / "main.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert (r.returncode, r.stdout) == (0, "ok\n"), (r.returncode, r.stdout)
