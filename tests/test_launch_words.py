"""Which word of pinned memory a selection of a shape goes by (csrc/launch_words.hpp), on the CPU."""

import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "evox_amd", "csrc")

PROGRAM = r"""
#include "launch_words.hpp"
#include <initializer_list>
#include <cstdio>
int main() {
  std::printf("%d\n", evx::kWordsPerMeaning * evx::kLaunchWords);
  for (int meaning = 0; meaning < evx::kLaunchWords; ++meaning)
    for (long long n : {1ll, 100ll, 57344ll, 57351ll, 90112ll, 200003ll, 0x7FFFFF00ll})
      for (int m = 1; m <= 16; ++m) std::printf("%d %d\n", meaning, evx::launch_word((evx::LaunchWord)meaning, n, m));
}
"""


def test_no_word_has_two_meanings(tmp_path):
    """A word that says of one shape that its last front is none for the sorted runs must not say of another, seven rows
    larger, that front 0 fell short."""
    (tmp_path / "words.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, "-o", str(tmp_path / "words"), str(tmp_path / "words.cpp")], check=True)
    lines = subprocess.run([str(tmp_path / "words")], capture_output=True, text=True, check=True, timeout=60).stdout.split("\n")
    total, meanings = int(lines[0]), {}
    for line in lines[1:-1]:
        meaning, word = map(int, line.split())
        assert 0 <= word < total
        assert meanings.setdefault(word, meaning) == meaning
    assert len(meanings) == total  # (sixteen objectives reach every word)
