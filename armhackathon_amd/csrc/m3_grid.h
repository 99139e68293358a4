// The token-grid layouts of the Mamba-3 scans (m3_grid.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace armscan {

constexpr int kGridSections = 8;

// One tensor of a grid: `planes` planes of H x W cells of `units` floats, and its row-major
// and column-major orderings stacked, (2 planes, H W, units).
struct GridSection {
  const float* src;
  float* dst;
  long long planes;
  int units;
  int vec;  // set by grid_to_views: 16-byte pieces
};
hipError_t grid_to_views(const GridSection* s, int n, int H, int W, hipStream_t st);
// out (batch, H, W, units) = scale (f + b of the row ordering + f + b of the column
// ordering), f and b (2 batch, H W, units); b may be null.
hipError_t views_to_grid(float* out, const float* f, const float* b, int batch, int H, int W,
                         int units, float scale, hipStream_t st);

}  // namespace armscan
