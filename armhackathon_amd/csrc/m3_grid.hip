// The token-grid layouts around the Mamba-3 scans (python/arm_scan/ss2d_mamba3.py: the
// row-major and column-major orderings of a grid stacked as sequences, and their outputs
// back on the grid), one kernel each way.
//
// Composed of torch ops the layouts are 16 copies and 3 sums of a few microseconds each, a
// strided copy and a concatenation per tensor, and the host needs longer to launch them
// than the GPU for the scans: 215 us at B2 28x28 H6 dv32 dqk64, of which the scans are 70.
// Here every tensor's two orderings leave in one launch (8.6 us there), and the four
// traversals meet in another (4.7 us): 95 us a call. B4 48x48: 485 -> 188 us, 18 and 7 of it.

#include <hip/hip_runtime.h>

#include <cstdint>

#include "m3_grid.h"

namespace armscan {

namespace {

struct Sections {
  GridSection s[kGridSections];
  long long first[kGridSections + 1];  // first unit of each section
  int n;
};

// Unit e of a section, in the order of its output: unit c of cell t of plane pl, the column
// ordering's planes after the row ordering's.
__global__ void __launch_bounds__(256) grid_to_views_kernel(Sections a, int H, int W) {
  const unsigned HW = (unsigned)H * W;
  const long long stride = (long long)gridDim.x * 256;
  for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < a.first[a.n]; e += stride) {
    int k = 0;
    while (e >= a.first[k + 1]) ++k;
    const GridSection& s = a.s[k];
    const long long rel = e - a.first[k];
    const long long cell = rel / s.units;
    const int c = (int)(rel - cell * s.units);
    const long long pl = cell / HW;
    const unsigned t = (unsigned)(cell - pl * HW);
    const bool col = pl >= s.planes;
    const unsigned from = col ? (t % H) * W + t / H : t;
    const long long src = ((pl - (col ? s.planes : 0)) * HW + from) * s.units + c;
    if (s.vec) reinterpret_cast<float4*>(s.dst)[rel] = reinterpret_cast<const float4*>(s.src)[src];
    else s.dst[rel] = s.src[src];
  }
}

// out = scale (f_rows + b_rows + f_cols + b_cols), added in that order; b null: one
// traversal an ordering. f and b (2 batch, H W, units).
template <typename V>
__global__ void __launch_bounds__(256) views_to_grid_kernel(V* __restrict__ out,
                                                            const V* __restrict__ f,
                                                            const V* __restrict__ b, int batch,
                                                            int H, int W, int units,
                                                            float scale) {
  const unsigned HW = (unsigned)H * W;
  const long long n = (long long)batch * HW * units, stride = (long long)gridDim.x * 256;
  for (long long e = (long long)blockIdx.x * 256 + threadIdx.x; e < n; e += stride) {
    const long long cell = e / units;
    const int c = (int)(e - cell * units);
    const long long bi = cell / HW;
    const unsigned t = (unsigned)(cell - bi * HW);
    const long long cols = ((batch + bi) * HW + (t % W) * H + t / W) * units + c;
    V v = f[e];
    if (b) v += b[e];
    v += f[cols];
    if (b) v += b[cols];
    out[e] = v * scale;
  }
}

unsigned grid_blocks(long long n) {
  const long long b = (n + 255) / 256;
  return (unsigned)(b < 1 ? 1 : b > 8192 ? 8192 : b);
}
bool a16(const void* q) { return ((uintptr_t)q & 15u) == 0; }

typedef float f4 __attribute__((ext_vector_type(4)));

}  // namespace

hipError_t grid_to_views(const GridSection* s, int n, int H, int W, hipStream_t st) {
  if (n < 1 || n > kGridSections) return hipErrorInvalidValue;
  Sections a{};
  a.n = n;
  for (int k = 0; k < n; ++k) {
    a.s[k] = s[k];
    a.s[k].vec = s[k].units % 4 == 0 && a16(s[k].src) && a16(s[k].dst);
    if (a.s[k].vec) a.s[k].units /= 4;
    a.first[k + 1] = a.first[k] + 2LL * s[k].planes * H * W * a.s[k].units;
  }
  hipLaunchKernelGGL(grid_to_views_kernel, dim3(grid_blocks(a.first[n])), dim3(256), 0, st, a, H,
                     W);
  return hipGetLastError();
}

hipError_t views_to_grid(float* out, const float* f, const float* b, int batch, int H, int W,
                         int units, float scale, hipStream_t st) {
  const bool vec = units % 4 == 0 && a16(out) && a16(f) && (!b || a16(b));
  const long long n = (long long)batch * H * W * units / (vec ? 4 : 1);
  if (vec)
    hipLaunchKernelGGL(views_to_grid_kernel<f4>, dim3(grid_blocks(n)), dim3(256), 0, st,
                       reinterpret_cast<f4*>(out), reinterpret_cast<const f4*>(f),
                       reinterpret_cast<const f4*>(b), batch, H, W, units / 4, scale);
  else
    hipLaunchKernelGGL(views_to_grid_kernel<float>, dim3(grid_blocks(n)), dim3(256), 0, st, out,
                       f, b, batch, H, W, units, scale);
  return hipGetLastError();
}

}  // namespace armscan
