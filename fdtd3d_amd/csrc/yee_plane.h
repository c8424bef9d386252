// Several steps of a 2D run in one launch (yee_plane.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "yee_kernels.h"

namespace yee {

// The most steps of a launch, the waves of a tile and the rows of a wave (FP64 holds half as many
// values per register).
constexpr int kPlaneSteps = 8;
constexpr int kPlaneWaves = 16;
#define PLANE_RW(T) (sizeof (T) == 4 ? 4 : 3)

// Tiles of a launch: columns of tiles, their count, tiles per XCD band, the margin of a tile and
// the steps to take (n <= margin).
struct PlaneGrid
{
  int ncol, ntile, per_xcd;
  int margin, n;
};

// Value of the hard source in every half step of a launch.
struct PlaneSource
{
  double v[kPlaneSteps][2];
};

template <typename T>
void launch_plane (int scheme, const StepArgs<T> &a, const PlaneGrid &g, const PlaneSource &src, hipStream_t stream);

}  // namespace yee
