"""How many workgroups peel a population by records and what their records hold (csrc/records.hpp), on the CPU."""

import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "evox_amd", "csrc")

PROGRAM = r"""
#define __host__
#define __device__
#include "records.hpp"
#include <cstdio>
int main() {
  const long long sizes[] = {1025, 32768, 32769, 65534, 65535, 150000, 163840, 163841, 170000, 200000, 262144};
  for (long long n : sizes)
    for (int m = 1; m <= 16; ++m) {
      const int sweepers = evx::record_sweepers(n, m);
      const bool wide = n > evx::kRecordsMaxRows;
      std::printf("%lld %d %d %d %lld\n", n, m, sweepers, evx::record_units(sweepers, wide ? evx::kRecUnitsWide : evx::kRecUnits),
                  (long long)evx::record_room(sweepers, wide));
    }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    where = tmp_path_factory.mktemp("records")
    (where / "records.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, "-o", str(where / "records"), str(where / "records.cpp")], check=True)
    lines = subprocess.run([str(where / "records")], capture_output=True, text=True, check=True, timeout=60).stdout.splitlines()
    return [tuple(int(v) for v in line.split()) for line in lines]


def test_records_fit_a_generation(plans):
    for n, m, sweepers, units, room in plans:
        assert sweepers * units <= (4096 if n > 65534 else 1024) and units & (units - 1) == 0
        assert sweepers + 1 <= 256 and -(-n // (sweepers * 8)) <= 256  # (256 rows per wave)


def test_large_fronts_keep_their_room(plans):
    """Fronts of uniform fitness with four objectives hold some 5000 rows at 150 000 and 6400 at 200 000: a record without
    room for its part of one sends every workgroup to the bitmaps in memory, in nearly every pass."""
    for n, m, sweepers, units, room in plans:
        if n > 65534:
            assert room >= (8064 if m >= 4 else 4960), (n, m, sweepers, room)
