// How the points of a hypervolume estimate are dealt to waves and workgroups.
#pragma once

#include <cstdint>

namespace evx {

// Points that a wave takes at a time, as scalar operands; one by one above 16 objectives.  (A step's values are in registers
// together: 8 objectives times 16 points no longer fit the 128 registers of a workgroup of 1024 threads, and went through
// scratch memory: 5000 x 8 against 20 000 samples, 1861 us, 100 with eight points.  From 9 objectives on the values are read
// objective by objective.)
constexpr int hv_step(int m) { return m > 16 ? 1 : (m == 8 ? 8 : 16); }

// Where 64 samples to a workgroup leave the device idle, the workgroups of the same samples are as many as fill it twice over
// (two of 1024 threads fit a compute unit), as far as every wave keeps eight steps: a wave alone pays the latency of every load
// itself.  Whole calls of the count with one workgroup per 64 samples and with this: 1 000 000 x 3 against 64 samples 3760 us, 42;
// against 10 000 3688, 2469; 100 000 x 17 against 1000 25 400, 914.  From some 65 000 samples on one part is all there is.
constexpr int64_t kHvFill = 4;        // workgroups per compute unit
constexpr int64_t kHvLeastSteps = 8;

struct HvSplit {
  unsigned threads;  // of a workgroup: its waves share the points of its 64 samples
  unsigned parts;    // workgroups that have the same 64 samples, and every parts-th turn of the waves each
};
constexpr HvSplit hv_split(int64_t n, int64_t n_sample, int step, int64_t cus) {
  int64_t waves = n_sample > (1ll << 28) ? 1 : (n_sample > 65536 ? 4 : 16);  // (a grid has less than 2^32 threads)
  const int64_t steps = (n + step - 1) / step, blocks = (n_sample + 63) / 64;
  if (waves > steps) waves = steps;
  int64_t parts = kHvFill * cus / blocks;
  const int64_t most = steps / (waves * kHvLeastSteps);
  if (parts > most) parts = most;
  if (parts < 1) parts = 1;
  return {(unsigned)(64 * waves), (unsigned)parts};
}

}  // namespace evx
