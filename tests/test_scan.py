"""The saturating count sums behind the cell list's overflow guard, on the
CPU: ions packed inside one cutoff make n^2 / 16384 units, past 32 bits from
6 million ions."""

import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "opendust_amd", "csrc")

# unit counts of the own-column entries of one column of n ions (groups of
# 128, 64-ion units), one entry in five as with four empty forward columns,
# added as launch_scan does: tiles of 1024, then the tile sums, then inside the
# tiles.  Prints the 64-bit total, the scan's, the largest offset error and
# what a plain 32-bit sum gives.
PROGRAM = r"""
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "od_scan.h"
using od::add_counts;
int main(int, char** v) {
  const int64_t n = atoll(v[1]);
  std::vector<int> cnt;
  for (int64_t t0 = 0; t0 < n; t0 += 128) {
    for (int k = 0; k < 4; ++k) cnt.push_back(0);
    cnt.push_back((int)((n - t0 + 63) / 64));
  }
  int64_t exact = 0, worst = 0;
  uint32_t wrapped = 0;
  int off = 0;
  for (size_t b = 0; b < cnt.size(); b += 1024) {
    int tile = 0, run = off;
    for (size_t i = b; i < b + 1024 && i < cnt.size(); ++i) {
      if (exact < od::COUNT_MAX && llabs(run - exact) > worst) worst = llabs(run - exact);
      tile = add_counts(tile, cnt[i]);
      run = add_counts(run, cnt[i]);
      exact += cnt[i];
      wrapped += (uint32_t)cnt[i];
    }
    off = add_counts(off, tile);
  }
  printf("%lld %d %lld %d\n", (long long)exact, off, (long long)worst, (int32_t)wrapped);
}
"""


@pytest.fixture(scope="module")
def packed_units(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("scan")
    (d / "scan.cpp").write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O2", "-I", CSRC, "-o", str(d / "scan"), str(d / "scan.cpp")], check=True)
    return lambda n: [int(w) for w in subprocess.run([str(d / "scan"), str(n)], check=True, capture_output=True,
                                                     text=True).stdout.split()]


# 5.93e6 ions: the last sum below 2^31; 8.4e6: past 2^32, where a wrapped sum
# is small and positive again; 2^28: the most a context takes
@pytest.mark.parametrize("n", [1, 129, 5_930_000, 6_000_000, 7_000_000, 8_400_000, 1 << 28])
def test_unit_sum_of_packed_ions_saturates(packed_units, n):
    limit = (1 << 31) - 1
    cap = 1_000_000_000  # the largest unit buffer
    exact, total, worst, wrapped = packed_units(n)
    assert total == min(exact, limit) and worst == 0
    assert (total > cap) == (exact > cap)
    if n == 6_000_000:
        assert wrapped < 0
    if n == 8_400_000:
        assert 0 < wrapped < cap < exact
