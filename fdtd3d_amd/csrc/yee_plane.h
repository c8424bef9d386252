// Several steps of a 2D or 1D run in one launch (yee_plane.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "yee_kernels.h"

namespace yee {

// The most steps of a launch, the rows of a wave (FP64 holds half as many values per register) and
// the waves of a tile.
constexpr int kPlaneSteps = 8;
#define PLANE_RW(T) (sizeof (T) == 4 ? 4 : 3)
constexpr int kPlaneWaves = 16, kPlaneWavesSmall = 8;

// Tiles of a launch: columns of tiles, their count, tiles per XCD band, the margin of a tile and
// the steps to take (n <= margin).
struct PlaneGrid
{
  int ncol, ntile, per_xcd;
  int margin, n;
  int waves;
};

// The tiles of n steps on a plane of nr x nc cells: kPlaneWavesSmall waves while the device's ncu
// compute units take all such tiles at once (a step of a tile then takes half as long: 100^2 FP64
// 2.5 us a step with 16 waves, 1.8 with 8), kPlaneWaves where tiles run in turns (less of a larger
// tile is margin).
template <typename T>
PlaneGrid plane_grid (int64_t nr, int64_t nc, int n, int ncu)
{
  PlaneGrid g {};
  g.n = n;
  g.margin = n;
  const int64_t cols = 64 - 2 * n;
  g.ncol = (int) ((nc - 2 + cols - 1) / cols);
  int64_t nt = 0;
  for (int w : { kPlaneWavesSmall, kPlaneWaves })
  {
    g.waves = w;
    const int64_t rows = PLANE_RW (T) * w - 2 * n;
    nt = (nr - 2 + rows - 1) / rows * (int64_t) g.ncol;
    if (nt <= ncu) break;
  }
  g.ntile = nt > (int64_t) 1 << 28 ? -1 : (int) nt;   // -1: too large for one launch
  g.per_xcd = (int) ((nt + 7) / 8);
  return g;
}

// Value of the hard source in every half step of a launch.
struct PlaneSource
{
  double v[kPlaneSteps][2];
};

// Fills a.pfac (arrays of pairs) for the components the scheme has.
template <typename T>
void launch_plane_factors (int scheme, const StepArgs<T> &a, hipStream_t stream);

// Tiles of a batched TMz sweep: 40 owned rows; the steps of a launch (the margin), the waves of a tile
// and the rows of a wave.  FP32: 8 waves of 7 rows (118 registers, two tiles a compute unit): 64
// simulations of 5.7e7 cells take 196 us a step, 242 with 14 waves of 4 rows (one tile a unit), 214
// with 12 of 4 and a margin of 4, 268 with 8 of 6 and a margin of 4.  FP64: 16 of 3 with a margin of
// 4, half the steps for less margin, which its lower tiles make dearer.
constexpr int kBatchRows = 40;
#define BATCH_STEPS(T) (sizeof (T) == 4 ? 8 : 4)
#define BATCH_WAVES(T) (sizeof (T) == 4 ? 8 : 16)
#define BATCH_RW(T) (sizeof (T) == 4 ? 7 : 3)

// n <= BATCH_STEPS steps of the simulations of a tile table (sim, x0, y0, -): from the step and buffer
// in state[sim], `off` steps and `flip` buffers on.
template <typename T>
void launch_batch_plane (const StepArgs<T> *sims, const int4 *tiles, int ntiles, const int *state, const T *src_tab,
                         int src_len, int off, int flip, int n, hipStream_t stream);

// Value of the hard source in every half step of a launch of a 1D run.
struct LineSource
{
  double v[kIncSteps][2];
};

// n <= kIncSteps steps of a 1D run (scheme YEE_SCHEME_EXHY .. EZHY).
template <typename T>
void launch_line (int scheme, const StepArgs<T> &a, int n, const LineSource &src, hipStream_t stream);

template <typename T>
void launch_plane (int scheme, const StepArgs<T> &a, const PlaneGrid &g, const PlaneSource &src, hipStream_t stream);

}  // namespace yee
