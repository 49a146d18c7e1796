// How many workgroups peel a population from memory by records (peel_records_kernel in peel.hpp), and how many rows a record
// holds.  Host and device.
#pragma once

#include <cstdint>

namespace evx {

constexpr int kRecordsMaxRows = 65534;       // largest population whose record units hold three 16-bit slots
constexpr int kRecordsMaxRowsWide = 262144;  // largest population peeled with the record protocol at all (two
                                             // 24-bit slots per unit; 128 blocks of 8 waves own 256 rows per wave)
constexpr int kRecUnits = 1024;  // units of one generation = sweepers x units per record
// Populations of 65 535 rows and more (the wide layout: two slots per unit) have fronts of thousands of rows, and a
// workgroup whose rows of a front do not fit its record sends everybody to the bitmaps in memory for that pass
// (200 000 x 3: 2000 rows a front, 128 sweepers with room for 15 each).  Their generations hold four times the
// units: room for 63 rows per workgroup with 128 sweepers, for 31 with 160.
constexpr int kRecUnitsWide = 4 * kRecUnits;

// Units of a record: the largest power of two that gives every sweeper a record (what belongs to which unit is told from
// the low bits of its index).
__host__ __device__ constexpr int record_units(int sweepers, int generation_units) {
  int units = 1;
  while (units * 2 * sweepers <= generation_units) units *= 2;
  return units;
}
// Rows of a front that the records of `sweepers` workgroups hold, when they are spread evenly.
constexpr int64_t record_room(int sweepers, bool wide) {
  const int units = record_units(sweepers, wide ? kRecUnitsWide : kRecUnits);
  return (int64_t)sweepers * (wide ? 1 + 2 * (units - 1) : 2 + 3 * (units - 1));
}

// Sweeping workgroups by size: 64 up to 32 768 rows, 128 above (20 000 rows: 221 us per selection with 64, 225 with 128,
// 228 with 32, 238 with 192; between 1200 and 6000 rows the count hardly matters).  Above five times that 160 with up to
// three objectives: more waves for the rescans outweigh the longer exchange there, but 160 is no power of two, its records
// have half the room (31 rows), and fronts of four objectives and more go through the bitmaps for it.  128 / 160, us per
// selection of half the rows, uniform fitness: x 3 60 000 477 / 550, 164 000 1139 / 1090, 200 003 1492 / 1397, 260 000
// 2195 / 2179;  x 4 150 000 882 / 898, 170 000 1034 / 1062, 200 000 1321 / 1357, 260 000 2016 / 2098;  x 5 170 000
// 1178 / 1196, 200 000 1518 / 1498;  x 8 200 000 1568 / 1564.
constexpr int record_sweepers(int64_t n, int m) { return n <= 32768 ? 64 : n <= 163840 || m > 3 ? 128 : 160; }

}  // namespace evx
