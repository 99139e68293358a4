// The Mamba-1 mixer's depthwise causal convolution on gfx950, the step before the scan
// in Hugging Face's MambaMixer (transformers modeling_mamba.py causal_conv1d_fn; the
// reference runs it upstream, python/arm_scan/patch.py patches only the scan):
//
//   y[b, d, t] = act(bias[d] + sum_{k < K} w[d, k] * x[b, d, t - (K-1) + k]),  x[t < 0] = 0
//
// x is any strided (batch, dim, len) view. The mixer hands over the first half of its
// in_proj output, (batch, len, 2*dim) storage, so channels are the contiguous axis.
// y is written (batch, dim, len) contiguous, the layout F.conv1d returns. The
// convolution is a transpose as well: a block stages a tile of kConvT + K - 1 steps x
// kConvD channels through LDS. It reads the tile along channels, the contiguous axis of
// such views, and writes along time.

#include <hip/hip_runtime.h>

#include <cstdint>

#include "scan_common.h"
#include "scan_launch.h"

namespace armscan {

namespace {

constexpr int kConvD = 64;        // channels per tile
constexpr int kConvT = 64;        // steps per tile
constexpr int kConvMaxK = 8;      // widest filter served
constexpr int kConvThreads = 256;

__global__ void __launch_bounds__(kConvThreads) causal_conv_kernel(CausalConv p) {
  __shared__ float tile[(kConvT + kConvMaxK - 1) * (kConvD + 1)];  // [step][channel], padded
  const int K = p.width;
  const long long b = blockIdx.z;
  const int d0 = blockIdx.y * kConvD;
  const long long t0 = (long long)blockIdx.x * kConvT;
  const int rows = kConvT + K - 1;  // steps t0-(K-1) .. t0+kConvT-1
  const float* xb = p.x + b * p.xs[0];
  if (p.vec) {
    // unit channel stride, 16-byte aligned rows: four channels per load
    for (int e = threadIdx.x; e < rows * (kConvD / 4); e += kConvThreads) {
      const int r = e / (kConvD / 4), c = 4 * (e - r * (kConvD / 4));
      const long long t = t0 - (K - 1) + r;
      const int d = d0 + c;
      float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (t >= 0 && t < p.len && d < p.dim)  // dim % 4 == 0: the piece is whole
        v = *reinterpret_cast<const float4*>(xb + d + t * p.xs[2]);
      float* row = tile + r * (kConvD + 1) + c;
      row[0] = v.x; row[1] = v.y; row[2] = v.z; row[3] = v.w;
    }
  } else {
    for (int e = threadIdx.x; e < rows * kConvD; e += kConvThreads) {
      const int r = e / kConvD, c = e - r * kConvD;
      const long long t = t0 - (K - 1) + r;
      const int d = d0 + c;
      float v = 0.0f;
      if (t >= 0 && t < p.len && d < p.dim) v = xb[(long long)d * p.xs[1] + t * p.xs[2]];
      tile[r * (kConvD + 1) + c] = v;
    }
  }
  __syncthreads();
  if (p.out_tm) {
    // (batch, len, dim) storage: consecutive lanes take consecutive channels, and a
    // thread keeps one channel (kConvThreads is a multiple of kConvD), whose taps and
    // bias it loads once
    static_assert(kConvThreads % kConvD == 0, "a thread keeps its channel");
    const int c = threadIdx.x % kConvD;
    const int d = d0 + c;
    if (d >= p.dim) return;  // no barrier follows
    float wr[kConvMaxK];
#pragma unroll
    for (int k = 0; k < kConvMaxK; ++k) wr[k] = k < K ? p.w[(long long)d * K + k] : 0.0f;
    const float bv = p.bias ? p.bias[d] : 0.0f;
    for (int r = threadIdx.x / kConvD; r < kConvT; r += kConvThreads / kConvD) {
      const long long t = t0 + r;
      if (t >= p.len) break;
      float acc = bv;
#pragma unroll
      for (int k = 0; k < kConvMaxK; ++k)
        if (k < K) acc = fmaf(wr[k], tile[(r + k) * (kConvD + 1) + c], acc);
      if (p.silu) acc = silu_fast(acc);
      p.out[(b * p.len + t) * p.dim + d] = acc;
    }
    return;
  }
  // (batch, dim, len): a thread keeps one step (kConvThreads is a multiple of kConvT)
  // and walks the channels, each wave on one channel, so taps and bias are uniform
  static_assert(kConvThreads % kConvT == 0, "a thread keeps its step");
  const int r = threadIdx.x % kConvT;
  const long long t = t0 + r;
  if (t >= p.len) return;  // no barrier follows
  for (int c = threadIdx.x / kConvT; c < kConvD; c += kConvThreads / kConvT) {
    const int d = d0 + c;
    if (d >= p.dim) break;
    float acc = p.bias ? p.bias[d] : 0.0f;
#pragma unroll
    for (int k = 0; k < kConvMaxK; ++k)
      if (k < K) acc = fmaf(p.w[(long long)d * K + k], tile[(r + k) * (kConvD + 1) + c], acc);
    if (p.silu) acc = silu_fast(acc);
    p.out[(b * p.dim + d) * p.len + t] = acc;
  }
}

// Width 4, time-major in and out by 16-byte pieces (the mixer's call): nothing is turned, so
// a thread takes four channels down T steps, their window of three in registers. A wave reads
// and writes 1 KB runs; each run of T steps reads three more. All T + 3 loads are independent
// and in flight at once, where the tile kernel's two phases wait at a barrier: B8 D1536 L2048
// 50 -> 40 us (5.0 TB/s, the rate of a large copy), B4 L1531 23 -> 19, B1 L77 7.3 -> 3.4. T 16
// for large calls (19% more loads, from L2), 4 where 16 would leave the chip idle.
template <int T>
__global__ void __launch_bounds__(kConvThreads) causal_conv_tm4_kernel(CausalConv p) {
  const int quads = p.dim / 4;
  const long long e = (long long)blockIdx.x * kConvThreads + threadIdx.x;
  const long long run = e / quads;  // run of T steps: batch * runs a row
  const int d = 4 * (int)(e - run * quads);
  const long long runs = (p.len + T - 1) / T;
  const long long b = run / runs, t0 = (run - b * runs) * T;
  if (b >= p.batch) return;
  const float* x = p.x + b * p.xs[0] + d;
  float4 v[T + 3];
#pragma unroll
  for (int i = 0; i < T + 3; ++i) {
    const long long t = t0 - 3 + i;
    v[i] = t >= 0 && t < p.len ? *reinterpret_cast<const float4*>(x + t * p.xs[2])
                               : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  }
  float4 w[4];  // tap k of the four channels
  const float* wd = p.w + 4LL * d;
  w[0] = make_float4(wd[0], wd[4], wd[8], wd[12]);
  w[1] = make_float4(wd[1], wd[5], wd[9], wd[13]);
  w[2] = make_float4(wd[2], wd[6], wd[10], wd[14]);
  w[3] = make_float4(wd[3], wd[7], wd[11], wd[15]);
  const float4 bias = p.bias ? make_float4(p.bias[d], p.bias[d + 1], p.bias[d + 2], p.bias[d + 3])
                             : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  float* out = p.out + (b * p.len + t0) * p.dim + d;
#pragma unroll
  for (int i = 0; i < T; ++i) {
    if (t0 + i >= p.len) break;
    float4 a = bias;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      a.x = fmaf(w[k].x, v[i + k].x, a.x);
      a.y = fmaf(w[k].y, v[i + k].y, a.y);
      a.z = fmaf(w[k].z, v[i + k].z, a.z);
      a.w = fmaf(w[k].w, v[i + k].w, a.w);
    }
    if (p.silu) a = make_float4(silu_fast(a.x), silu_fast(a.y), silu_fast(a.z), silu_fast(a.w));
    *reinterpret_cast<float4*>(out + (long long)i * p.dim) = a;
  }
}

// The decode step of the mixer's width, 4: a window is one 16-byte piece, read and written
// whole (by single floats: 4.8 -> 3.5 us at batch 128, D 1536, 3.3 -> 2.3 at batch 1).
__global__ void __launch_bounds__(kConvThreads) causal_conv_step4_kernel(CausalConvStep p) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;  // b * dim + d
  if (i >= (long long)p.batch * p.dim) return;
  const long long b = i / p.dim, d = i - b * p.dim;
  float4* s = reinterpret_cast<float4*>(p.state) + i;
  const float4 old = *s, w = reinterpret_cast<const float4*>(p.w)[d];
  const float x = p.x[b * p.xs[0] + d * p.xs[1]];
  float acc = p.bias ? p.bias[d] : 0.0f;
  acc = fmaf(w.x, old.y, acc);
  acc = fmaf(w.y, old.z, acc);
  acc = fmaf(w.z, old.w, acc);
  acc = fmaf(w.w, x, acc);
  *s = make_float4(old.y, old.z, old.w, x);
  if (p.silu) acc = silu(acc);
  p.out[i] = acc;
}

// One decode step of any width: thread (b, d) shifts its window of the conv state left by
// one, appends the new input and writes act(bias + w . window).
__global__ void __launch_bounds__(kConvThreads) causal_conv_step_kernel(CausalConvStep p) {
  const long long i = (long long)blockIdx.x * kConvThreads + threadIdx.x;  // b * dim + d
  if (i >= (long long)p.batch * p.dim) return;
  const long long b = i / p.dim, d = i - b * p.dim;
  float* s = p.state + i * p.width;
  const float* w = p.w + d * p.width;
  const float x = p.x[b * p.xs[0] + d * p.xs[1]];
  float acc = p.bias ? p.bias[d] : 0.0f;
  for (int k = 0; k < p.width; ++k) {
    const float v = k + 1 < p.width ? s[k + 1] : x;
    s[k] = v;
    acc = fmaf(w[k], v, acc);
  }
  if (p.silu) acc = silu(acc);
  p.out[i] = acc;
}

}  // namespace

hipError_t causal_conv1d_step(const CausalConvStep& p, hipStream_t st) {
  const long long rows = (long long)p.batch * p.dim;
  const long long blocks = (rows + kConvThreads - 1) / kConvThreads;
  if (blocks <= 0 || blocks > 0x7fffffffLL || p.width < 1) return hipErrorInvalidValue;
  if (p.width == 4 && (((uintptr_t)p.state | (uintptr_t)p.w) & 15u) == 0) {
    // few rows: blocks of one wave, so that they spread over the CUs
    const int threads = rows < 65536 ? 64 : kConvThreads;
    hipLaunchKernelGGL(causal_conv_step4_kernel, dim3((unsigned)((rows + threads - 1) / threads)),
                       dim3(threads), 0, st, p);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(causal_conv_step_kernel, dim3((unsigned)blocks), dim3(kConvThreads), 0,
                     st, p);
  return hipGetLastError();
}

hipError_t causal_conv1d(const CausalConv& p, hipStream_t st) {
  if (p.width < 1 || p.width > kConvMaxK || p.batch < 1 || p.dim < 1 || p.len < 1)
    return hipErrorInvalidValue;
  const long long tb = (p.len + kConvT - 1) / kConvT;
  if (tb > 0x7fffffffLL || p.batch > 65535 || (p.dim + kConvD - 1) / kConvD > 65535)
    return hipErrorInvalidValue;
  const dim3 grid((unsigned)tb, (unsigned)((p.dim + kConvD - 1) / kConvD), (unsigned)p.batch);
  CausalConv k = p;
  k.vec = p.xs[1] == 1 && p.dim % 4 == 0 && p.xs[0] % 4 == 0 && p.xs[2] % 4 == 0 &&
          ((uintptr_t)p.x & 15u) == 0;
  if (k.vec && p.out_tm && p.width == 4 && ((uintptr_t)p.out & 15u) == 0) {
    const long long row = (long long)p.batch * (p.dim / 4);  // threads a run of all rows
    const bool large = row * ((p.len + 15) / 16) >= 65536;   // a wave for every SIMD
    const long long n = row * ((p.len + (large ? 15 : 3)) / (large ? 16 : 4));
    const long long blocks = (n + kConvThreads - 1) / kConvThreads;
    if (blocks <= 0x7fffffffLL) {
      if (large)
        hipLaunchKernelGGL(causal_conv_tm4_kernel<16>, dim3((unsigned)blocks),
                           dim3(kConvThreads), 0, st, k);
      else
        hipLaunchKernelGGL(causal_conv_tm4_kernel<4>, dim3((unsigned)blocks),
                           dim3(kConvThreads), 0, st, k);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL(causal_conv_kernel, grid, dim3(kConvThreads), 0, st, k);
  return hipGetLastError();
}

}  // namespace armscan
