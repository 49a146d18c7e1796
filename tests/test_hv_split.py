"""How the points of a hypervolume estimate are dealt to waves and workgroups (csrc/hv_split.hpp), on the CPU."""

import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "evox_amd", "csrc")

PROGRAM = r"""
#include "hv_split.hpp"
#include <cstdio>
#include <initializer_list>
int main() {
  const long long sizes[] = {1, 15, 16, 17, 50, 100, 1001, 5003, 20000, 65536, 65537, 100000, 1000000, 0x7FFFFF00ll};
  for (long long n : sizes)
    for (long long samples : sizes)
      for (int m : {1, 3, 8, 17}) {
        const evx::HvSplit d = evx::hv_split(n, samples, evx::hv_step(m), 256);
        std::printf("%lld %lld %d %d %u %u\n", n, samples, m, evx::hv_step(m), d.threads, d.parts);
      }
}
"""


@pytest.fixture(scope="module")
def deals(tmp_path_factory):
    where = tmp_path_factory.mktemp("split")
    (where / "split.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, "-o", str(where / "split"), str(where / "split.cpp")], check=True)
    lines = subprocess.run([str(where / "split")], capture_output=True, text=True, check=True, timeout=60).stdout.splitlines()
    return [tuple(int(v) for v in line.split()) for line in lines]


def test_every_deal_can_be_launched(deals):
    for n, samples, m, step, threads, parts in deals:
        assert threads % 64 == 0 and 64 <= threads <= 1024 and 1 <= parts <= 65535
        assert (samples + 63) // 64 * threads < 2**32
        assert threads // 64 * parts <= (n + step - 1) // step, "a wave without points"


def test_few_samples_still_fill_the_device(deals):
    """A workgroup per 64 samples alone leaves most compute units idle: the points are shared until the workgroups go round
    or a wave has only a few steps left."""
    for n, samples, m, step, threads, parts in deals:
        blocks = (samples + 63) // 64
        steps_per_wave = n / step / (threads // 64 * parts)
        assert blocks * parts >= 512 or steps_per_wave < 32, (n, samples, m, parts)
        assert parts == 1 or blocks * parts <= 1024
