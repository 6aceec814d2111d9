// What the two-step kernel's 32-bit buffer offsets reach. Plain C++.
#pragma once
#include <cstdint>

namespace wf {

// The offset of a lane without cells: it reads zeros and writes nothing, as long
// as no array is longer than OOB bytes.
constexpr uint32_t OOB = 0xfffffff0u;

// Whether every array of a grid is within reach: the 3N fields and the six 2-D
// metric tables, which lie in one array (longer than the fields on grids of one
// line of cells).
constexpr bool t2_in_reach(int64_t Nx, int64_t Ny, int64_t Nz, int elem) {
  const uint64_t fields = 3 * (uint64_t)Nx * (uint64_t)Ny * (uint64_t)Nz;
  const uint64_t tables = 2 * ((uint64_t)Ny * Nz + (uint64_t)Nx * Nz + (uint64_t)Nx * Ny);
  return fields * elem <= OOB && tables * elem <= OOB;
}

}  // namespace wf
