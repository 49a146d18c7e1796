"""The deal of the rows that a leaf of the first front leaves open (csrc/deal.hpp), on the CPU: threads in the place of the
waves, one of which answers as soon as it may while the others read the word as late as they can.  Every open row must be
asked exactly once."""

import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "evox_amd", "csrc")

PROGRAM = r"""
#define __host__
#define __device__
#include "deal.hpp"
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <thread>
#include <vector>

int main(int, char** argv) {
  const int waves = 4, early = std::atoi(argv[1]);
  const uint64_t rows = std::strtoull(argv[2], nullptr, 0);
  std::atomic<uint64_t> decided{0};
  std::atomic<int> asked[64] = {};
  std::mutex lock;
  std::condition_variable changed;
  int arrived = 0;
  bool answered = false;
  auto wave = [&](int w) {
    evx::deal_open_rows(
        w, waves,
        [&] {
          if (w != early) {  // late: after the early wave's first answer, if that comes before this read
            std::unique_lock<std::mutex> hold(lock);
            changed.wait_for(hold, std::chrono::milliseconds(300), [&] { return answered; });
          }
          return rows & ~decided.load();
        },
        [&] {
          std::unique_lock<std::mutex> hold(lock);
          ++arrived;
          changed.notify_all();
          changed.wait(hold, [&] { return arrived == waves; });
        },
        [&](int r) {
          ++asked[r];
          decided |= 1ull << r;
          std::lock_guard<std::mutex> hold(lock);
          answered = true;
          changed.notify_all();
        });
  };
  std::vector<std::thread> threads;
  for (int w = 0; w < waves; ++w) threads.emplace_back(wave, w);
  for (auto& t : threads) t.join();
  int wrong = 0;
  for (int r = 0; r < 64; ++r) wrong += asked[r] != (int)((rows >> r) & 1u);
  std::printf("%d\n", wrong);
  return wrong != 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    where = tmp_path_factory.mktemp("deal")
    source = where / "deal.cpp"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", CSRC, "-o", str(where / "deal"), str(source)], check=True)
    return str(where / "deal")


@pytest.mark.parametrize("early", [0, 3])
@pytest.mark.parametrize("rows", [0x1, 0xF, 0x1F, 0x8000000000000421, 0xFFFFFF])
def test_every_open_row_is_asked_once(program, rows, early):
    done = subprocess.run([program, str(early), hex(rows)], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, f"{done.stdout.strip()} rows were not asked exactly once"
