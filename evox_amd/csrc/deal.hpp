// Work dealt to the waves of a workgroup from a word in LDS that the same waves change while they work.
#pragma once

#include <cstdint>

namespace evx {

// The rows set in open() are dealt to `waves` waves by their position among them, and ask(row) is called for this wave's.
// ask may clear rows of the word that open reads, so every wave must hold the same word before the first of them asks: a wave
// that read later would count the positions differently, and a row could be no wave's.  barrier: of the whole workgroup.
template <class Open, class Barrier, class Ask>
__host__ __device__ inline void deal_open_rows(int wave, int waves, Open open, Barrier barrier, Ask ask) {
  const uint64_t rows = open();
  barrier();
  int turn = wave;  // rows until this wave's next one
  for (uint64_t todo = rows; todo != 0ull; todo &= todo - 1) {
    if (turn != 0) {
      --turn;
      continue;
    }
    turn = waves - 1;
    ask(__builtin_ctzll(todo));
  }
}

}  // namespace evx
