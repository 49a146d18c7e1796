// Where the words lie by which a selection chooses its launches (outcome_slot in api.hip).
#pragma once

#include <cstdint>

namespace evx {

// What a word is about; every meaning has words of its own.
enum LaunchWord {
  kWordLastFront = 0,  // selections of 4-byte fitness: the peel kernel ordered the last front (1) or left it (2)
  kWordBatch = 1,      // ... of several populations in a launch: what became of the first one's
  kWordWide = 2,       // those whose last front is ordered by the kernels of wide.hpp: it was small (1) or large (2)
  kWordFront0 = 3,     // whether front 0 alone held what was kept (GatherArgs::front0_note)
  kWordRuns = 4,       // above kMidArgsortRows rows: the last front was one for the sorted runs (1) or not (2)
  kLaunchWords = 5,
};
constexpr int kWordsPerMeaning = 16;  // shapes that share a word cost each other a guess, no more

constexpr int launch_word(LaunchWord meaning, int64_t n, int64_t m) {
  return (int)meaning * kWordsPerMeaning + (int)(((uint64_t)n * 31u + (uint64_t)m) % kWordsPerMeaning);
}

}  // namespace evx
