// fippi_heap.h -- how many workgroups the FIPPI cubature runs with.
#pragma once

#include <algorithm>
#include <cstddef>

namespace scuffx {

// regions of a heap: enough for the whole evaluation budget (1e6 points, 66 per
// split); its bytes: record, key and slot number per region
constexpr int kFippiCap = 15360;
constexpr size_t kFippiHeapBytes = (size_t)kFippiCap * (76 * sizeof(double) + sizeof(double) + sizeof(int));

// workgroups (each with a heap) for `jobs` jobs: up to four on each of 256 CUs,
// fewer so that `reserve` of the free memory is left, but at least an eighth
// of it is used (what the reserve is for may be held already)
inline int fippi_slots(long jobs, size_t free_bytes, size_t reserve)
{
  const size_t budget = std::max(free_bytes / 8, free_bytes > reserve ? free_bytes - reserve : (size_t)0);
  const long fit = (long)std::min<size_t>(budget / kFippiHeapBytes, 1024);
  return (int)std::max(1L, std::min(fit, jobs));
}

}  // namespace scuffx
