// The Mamba-3 mixer's front-end on gfx950 (apps/mamba3_lm/block.py:146-178): what
// sits between in_proj and the scan, in one kernel over the projection
//
//   proj (b, l, row_stride), columns [z | x | B | C | dd_dt | dd_A | trap | angles]
//   (block.py:113-118, the checkpoint's order)
//
//   dt   = softplus(dd_dt + dt_bias)                         -> (b, h, l)
//   adt  = min(-heavy_tail(dd_A), -A_floor) * dt              -> (b, h, l)
//          heavy_tail(x) = max(x, 0) + 1 / (1 - min(x, 0))    (block.py:52-62)
//   trap = trap, pre-sigmoid                                  -> (b, h, l)
//   k    = B * rsqrt(mean_n(B^2) + eps) * B_norm.weight       -> (b, l, r, g, n)
//   q    = C * rsqrt(mean_n(C^2) + eps) * C_norm.weight       (Q <- C, K <- B: block.py:187-197)
//
// z, x and the angles are not touched: the scan reads them in place from the
// projection by their strides (the angles with head stride 0, one set shared by every
// head as block.py:174 broadcasts them).
//
// Two kinds of block in one launch. Gate blocks take kTok consecutive tokens of one batch
// row; the gates go through LDS, 32 heads at a time, so that their head-major stores run
// along the sequence (kTok floats per head). Norm blocks take rows of B or C
// (d_state floats each), each row on as many lanes as it has four floats (32 at d_state
// 128), its sum of squares by shuffles, the rows of a wave loaded together.
//
// What bounds it is latency: about 10 KB a token-block. With both in one block of 32 tokens
// and a wave to each norm row, one after another, a prompt of 1024 tokens was 32 blocks of
// 16 dependent rows a wave: 26.5 us; now 5.0. B4 L4096: 38 -> 12.5 us (3.5 TB/s).

#include <hip/hip_runtime.h>

#include <cstdint>

#include "scan_common.h"
#include "scan_launch.h"

namespace armscan {

namespace {

constexpr int kTok = 32;
constexpr int kHeadGroup = 32;  // heads per pass through LDS
constexpr int kFrontThreads = 256;
constexpr int kNormPasses = 2;  // rows a lane group takes, loaded together

// Rows of B (k) and C (q): row r of the launch is row r % (2 rank groups) of token r / (2
// rank groups), on lpr lanes, by 16-byte pieces (VEC) or single floats.
template <bool VEC>
__device__ __forceinline__ void norm_rows(const M3Frontend& p, long long blk, int lpr) {
  const int n = p.d_state, rows = p.rank * p.groups;
  const int col_b = 2 * p.heads * p.headdim, col_c = col_b + rows * n;
  const int groups = kFrontThreads / lpr;  // lane groups of the block
  const int gi = threadIdx.x / lpr, lane = threadIdx.x % lpr;
  const long long total = 2LL * rows * p.batch * p.len;
  const long long r0 = blk * (groups * kNormPasses) + gi;
  const float* src[kNormPasses];
  float* dst[kNormPasses];
  const float* w[kNormPasses];
  float4 v[kNormPasses];
  float ss[kNormPasses];
#pragma unroll
  for (int k = 0; k < kNormPasses; ++k) {
    const long long r = r0 + k * groups;
    const long long rc = r < total ? r : total - 1;  // past the end: the last row, not stored
    const long long tok = rc / (2 * rows);
    const int rem = (int)(rc - tok * 2 * rows);
    const bool is_c = rem >= rows;
    const int rr = is_c ? rem - rows : rem;
    src[k] = p.proj + tok * p.row_stride + (is_c ? col_c : col_b) + rr * n;
    dst[k] = r < total ? (is_c ? p.q : p.k) + (tok * rows + rr) * (long long)n : nullptr;
    w[k] = is_c ? p.c_norm : p.b_norm;
    ss[k] = 0.0f;
    if constexpr (VEC) {
      v[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      for (int e = 4 * lane; e < n; e += 4 * lpr) {
        v[k] = *reinterpret_cast<const float4*>(src[k] + e);
        ss[k] = fmaf(v[k].x, v[k].x, ss[k]);
        ss[k] = fmaf(v[k].y, v[k].y, ss[k]);
        ss[k] = fmaf(v[k].z, v[k].z, ss[k]);
        ss[k] = fmaf(v[k].w, v[k].w, ss[k]);
      }
    } else {
      for (int e = lane; e < n; e += lpr) ss[k] = fmaf(src[k][e], src[k][e], ss[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < kNormPasses; ++k) {
    for (int d = lpr / 2; d > 0; d >>= 1) ss[k] += __shfl_xor(ss[k], d);
    if (dst[k] == nullptr) continue;  // the lane group alone: no shuffle follows across it
    const float rstd = 1.0f / sqrtf(ss[k] / (float)n + p.eps);
    if constexpr (VEC) {
      for (int e = 4 * lane; e < n; e += 4 * lpr) {
        // one piece a lane: still in registers
        const float4 x = n <= 4 * lpr ? v[k] : *reinterpret_cast<const float4*>(src[k] + e);
        const float4 g = *reinterpret_cast<const float4*>(w[k] + e);
        *reinterpret_cast<float4*>(dst[k] + e) =
            make_float4(x.x * rstd * g.x, x.y * rstd * g.y, x.z * rstd * g.z, x.w * rstd * g.w);
      }
    } else {
      for (int e = lane; e < n; e += lpr) dst[k][e] = src[k][e] * rstd * w[k][e];
    }
  }
}

template <bool VEC>
__global__ void __launch_bounds__(kFrontThreads)
m3_frontend_kernel(M3Frontend p, int gate_blocks, int lpr) {
  __shared__ float gl[3 * kHeadGroup * kTok];  // [3][head in group][token]: dt, adt, trap
  if ((int)blockIdx.x >= gate_blocks) {  // whole block: no barrier is reached
    norm_rows<VEC>(p, (long long)blockIdx.x - gate_blocks, lpr);
    return;
  }
  const int H = p.heads, L = p.len, rows = p.rank * p.groups;
  const int per = (L + kTok - 1) / kTok;  // gate blocks of a batch row
  const long long b = blockIdx.x / per;
  const int t0 = (int)(blockIdx.x - b * per) * kTok;
  const int ntok = L - t0 < kTok ? L - t0 : kTok;
  const float* base = p.proj + (b * L + t0) * p.row_stride;
  const int col_g = 2 * H * p.headdim + 2 * rows * p.d_state;

  constexpr int G = kHeadGroup;
  for (int h0 = 0; h0 < H; h0 += G) {  // block-uniform
    const int nh = H - h0 < G ? H - h0 : G;
    for (int e = threadIdx.x; e < ntok * nh; e += kFrontThreads) {
      const int j = e / nh, hh = e - j * nh, h = h0 + hh;
      const float* g = base + (long long)j * p.row_stride + col_g;
      const float dt = softplus(g[h] + p.dt_bias[h]);
      const float x = g[H + h];
      const float heavy = fmaxf(x, 0.0f) + 1.0f / (1.0f - fminf(x, 0.0f));
      gl[hh * kTok + j] = dt;
      gl[(G + hh) * kTok + j] = fminf(-heavy, -p.a_floor) * dt;
      gl[(2 * G + hh) * kTok + j] = g[2 * H + h];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < nh * ntok; e += kFrontThreads) {
      const int hh = e / ntok, j = e - hh * ntok;
      const long long o = (b * H + h0 + hh) * L + t0 + j;
      p.dt[o] = gl[hh * kTok + j];
      p.adt[o] = gl[(G + hh) * kTok + j];
      p.trap[o] = gl[(2 * G + hh) * kTok + j];
    }
    __syncthreads();  // gl is rewritten by the next group
  }
}

}  // namespace

hipError_t m3_frontend(const M3Frontend& p, hipStream_t st) {
  if (p.len <= 0 || p.batch <= 0 || p.heads <= 0) return hipErrorInvalidValue;
  const int n = p.d_state, rows = p.rank * p.groups;
  auto a16 = [](const void* q) { return ((uintptr_t)q & 15u) == 0; };
  // 16-byte pieces: every row of B and C (they start 2 heads headdim floats in), the
  // weights and the outputs on 16-byte bases
  const bool vec = n % 4 == 0 && p.row_stride % 4 == 0 && 2LL * p.heads * p.headdim % 4 == 0 &&
                   a16(p.proj) && a16(p.q) && a16(p.k) && a16(p.b_norm) && a16(p.c_norm);
  // lanes a row: the power of two that holds it four floats a lane, at most a wave. Single
  // floats too: a wave to each short row left most of its lanes idle and the chip dispatching
  // blocks of eight rows (2 heads, d_state 16, 262144 tokens of 298 floats: 146 -> 38 us).
  int lpr = 64;
  while (lpr > 1 && 4 * (lpr / 2) >= n) lpr /= 2;
  const long long gates = (long long)p.batch * ((p.len + kTok - 1) / kTok);
  const long long per_block = (kFrontThreads / lpr) * kNormPasses;
  const long long total = 2LL * rows * p.batch * p.len;
  const long long blocks = gates + (total + per_block - 1) / per_block;
  if (blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  if (vec)
    hipLaunchKernelGGL(m3_frontend_kernel<true>, dim3((unsigned)blocks), dim3(kFrontThreads), 0,
                       st, p, (int)gates, lpr);
  else
    hipLaunchKernelGGL(m3_frontend_kernel<false>, dim3((unsigned)blocks), dim3(kFrontThreads), 0,
                       st, p, (int)gates, lpr);
  return hipGetLastError();
}

}  // namespace armscan
