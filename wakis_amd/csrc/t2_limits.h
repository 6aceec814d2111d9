// What the two-step kernel's 32-bit buffer offsets reach. Plain C++.
#pragma once
#include <cstdint>

namespace wf {

// The offset of a lane without cells: it reads zeros and writes nothing, as long
// as no array is longer than OOB bytes.
constexpr uint32_t OOB = 0xfffffff0u;

// Whether the 3N arrays of a grid of N cells are within reach. The six 2-D metric
// tables, in one array, then are too: with at least two cells per axis they are
// no longer than a field.
constexpr bool t2_in_reach(int64_t N, int elem) { return 3 * (uint64_t)N * elem <= OOB; }

}  // namespace wf
