// Device 3D Delaunay tetrahedralisation, one vertex star per wave
// (stars3d.hip).
#pragma once

#include <cstdint>
#include <vector>

#include "common.h"

namespace smk {

// Why a build is left to the host (the kernels' status word uses the first
// five).
enum StarLeft {
  kLeftNot = 0,
  kLeftInput = 1,       // too few or many points, a flat set, coordinates out of range
  kLeftUnresolved = 2,  // a predicate beyond the exact stage
  kLeftPool = 3,        // more link triangles than the pool holds
  kLeftCells = 4,       // more cells than the output holds
  kLeftUncertain = 5,   // too many stars in need of exact predicates
  kLeftCrowded = 6,     // too many points to a cell of the search grid
  kLeftHubs = 7,        // too many large stars, or theirs could not be settled
  kLeftMemory = 8       // no memory for the scratch
};

// Scratch of the device build (one per handle, grown to its largest point
// set: about 0.6 kB a point).
struct StarScratch {
  void *mem = nullptr;
  size_t bytes = 0;
  size_t max_bytes = SIZE_MAX;  // builds that need more go to the host
  int32_t *h_status = nullptr;  // pinned
  int skip = 0;                 // builds left to the host after a failed one
  int left = kLeftNot;          // why the last build it looked at was left
};

void stars_free(StarScratch *s);

// Fewest points the device build takes on.  Its launches and the longest
// chain of dependent insertions take 0.5-0.7 ms whatever the size; the
// host's serial build takes 2 us a point (100 points: 0.2 ms against 0.65;
// 1000: 2.1 against 0.9).
constexpr int64_t kStarMinPoints = 512;

// The finite Delaunay tetrahedra of the n points p (device, (n, 3) FP64) to
// `tet` (device, room for cap cells): the same cells in the same order as
// sm_host_delaunay3d.  `spacing` is a typical distance between neighbouring
// points (any positive value is correct; it sizes the search grid);
// host_threads is the number of threads the host build would take.
// Synchronises the stream.  *done is false when the device leaves the build
// to the host (too few points, points in one plane, predicates its exact
// stage cannot settle, too many uncertain ones, very large stars or points to
// a cell of its grid, no memory for the scratch); nothing is written then that
// the host build does not replace.
int device_delaunay3d(StarScratch *sc, const double *p, int64_t n, double spacing,
                      int host_threads, int32_t *tet, int64_t cap, int64_t *count, bool *done,
                      hipStream_t s);

}  // namespace smk
