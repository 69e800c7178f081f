"""CPU: how the triangle / edge emptiness lists what its first phase leaves,
compiled from the library's header.  From 2^31 simplices on an id needs the
bit that marks an untested entry: then nothing is marked and the second phase
takes every entry as an id."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cstdio>
#include <initializer_list>
#include "pac_phases.h"
using namespace pac;
int main() {
  const int64_t sizes[] = {1, kPackItems - 1, kPackItems, 1ll << 24,
                           (1ll << 31) - 1, 1ll << 31, (1ll << 31) + 1,
                           (1ll << 32) - 2};
  for (int64_t n : sizes)
    for (int marks = 0; marks < 2; ++marks)
      for (int budget : {0, 6}) {
        const LowPhases p = low_phases(marks != 0, n, budget);
        int bad = 0;
        for (int64_t q : {(int64_t)0, n / 2, n - 1}) {
          const uint32_t id = (uint32_t)q;
          bad += left_id(id, p.whole) != id;
          bad += left_tested(id, p.whole, budget) != budget;
          if (p.pack) {
            bad += left_id(id | p.whole, p.whole) != id;
            bad += left_tested(id | p.whole, p.whole, budget) != 0;
          }
        }
        std::printf("%lld %d %d %d %d\n", (long long)n, marks, budget,
                    (int)p.pack, bad);
      }
}
"""


@pytest.fixture(scope="module")
def rows(tmp_path_factory):
    d = tmp_path_factory.mktemp("phases")
    (d / "probe.cpp").write_text(SRC)
    csrc = os.path.join(ROOT, "parallelac-xmp_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-I", csrc, str(d / "probe.cpp"),
                    "-o", str(d / "probe")], check=True)
    out = subprocess.run([str(d / "probe")], check=True, capture_output=True,
                         text=True).stdout
    return [tuple(map(int, line.split())) for line in out.splitlines()]


def test_every_id_survives_the_list(rows):
    assert len(rows) == 32 and all(bad == 0 for *_, bad in rows)


def test_packed_where_ids_leave_the_bit(rows):
    for n, marks, budget, pack, _ in rows:
        assert pack == (marks and budget > 0 and (1 << 17) <= n <= (1 << 31))
