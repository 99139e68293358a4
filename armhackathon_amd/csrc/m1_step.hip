// Mamba-1 decode: one step of the selective scan with the recurrent state updated
// in place, the single-token path of a generation loop (transformers
// modeling_mamba.py mamba_selective_state_update; the reference leaves it to upstream,
// README.md:320-322). Per (batch, channel) and state n:
//
//   dt = softplus(dt + bias) (when asked);  h_n <- exp(dt A_n) h_n + dt B_n x
//   y = sum_n C_n h_n + D x ;  y *= silu(z)
//
// the one-step case of scalar::scan (kernel/arm-scan-core/src/scalar.rs:11-89) with
// h0 = last_state = the state. The per-row inputs are given by strides, as a decoder hands
// them over (views of its projections). The states of a (batch, channel) row are the bytes
// that count (64 read and 64 written at N 16, of 150 in all): memory-bound for a large
// batch, one latency of dependent loads for a small one.

#include <hip/hip_runtime.h>

#include <cstdint>

#include "scan_common.h"
#include "scan_launch.h"

namespace armscan {

namespace {

constexpr int kStepThreads = 256;

// N a multiple of 4 with 16-byte aligned state and A: Q lanes to a row (a power of two
// dividing N / 4, at most 16), each taking every Q-th 16-byte piece of the row's states, so
// that a wave's loads and stores are contiguous (N 16: four lanes, 16 rows a wave), and the
// row's y summed over its lanes by shuffles. One thread a row moved 4 bytes of each of 64
// rows 64 bytes apart per instruction, and a row's loads waited for one another: batch 128,
// D 1536, N 16 28.6 -> 9.1 us (3.1 TB/s), batch 1 10.8 -> 3.4 us. VB: B and C by 16-byte
// pieces too (unit state stride, aligned).
template <bool VB>
__global__ void __launch_bounds__(kStepThreads) m1_step_vec_kernel(M1Step p, int Q) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long i = e / Q;  // b * dim + d
  const int q = (int)(e & (Q - 1));
  const bool on = i < (long long)p.batch * p.dim;  // whole rows: Q divides the block
  const long long r = on ? i : 0;
  const long long b = r / p.dim, d = r - b * p.dim;
  const float x = p.x[b * p.xs[0] + d * p.xs[1]];
  float dt = p.dt[b * p.dts[0] + d * p.dts[1]] + (p.bias ? p.bias[d] : 0.0f);
  const float z = p.z ? p.z[b * p.zs[0] + d * p.zs[1]] : 0.0f;
  const float skip = p.D ? p.D[d] : 0.0f;
  float4* h = reinterpret_cast<float4*>(p.state + r * p.N);
  const float4* A = reinterpret_cast<const float4*>(p.A + d * p.N);
  const float* B = p.B + b * p.Bs[0];
  const float* C = p.C + b * p.Cs[0];
  if (p.softplus) dt = softplus(dt);
  const float dx = dt * x;
  float y = 0.0f;
  for (int k = q; k < p.N / 4; k += Q) {
    const float4 h4 = h[k], a4 = A[k];
    const float hv[4] = {h4.x, h4.y, h4.z, h4.w}, av[4] = {a4.x, a4.y, a4.z, a4.w};
    float bv[4], cv[4], hn[4];
    if constexpr (VB) {
      const float4 b4 = reinterpret_cast<const float4*>(B)[k];
      const float4 c4 = reinterpret_cast<const float4*>(C)[k];
      bv[0] = b4.x; bv[1] = b4.y; bv[2] = b4.z; bv[3] = b4.w;
      cv[0] = c4.x; cv[1] = c4.y; cv[2] = c4.z; cv[3] = c4.w;
    } else {
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        bv[m] = B[(4 * k + m) * p.Bs[1]];
        cv[m] = C[(4 * k + m) * p.Cs[1]];
      }
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      hn[m] = fmaf(fexp(dt * av[m]), hv[m], dx * bv[m]);
      y = fmaf(cv[m], hn[m], y);
    }
    if (on) h[k] = make_float4(hn[0], hn[1], hn[2], hn[3]);
  }
  for (int m = 1; m < Q; m <<= 1) y += __shfl_xor(y, m, 16);
  if (!on || q != 0) return;
  if (p.D) y = fmaf(skip, x, y);
  if (p.z) y *= silu(z);
  p.out[i] = y;
}

// Any N, alignment and strides: one thread a row.
__global__ void __launch_bounds__(kStepThreads) m1_step_kernel(M1Step p) {
  const long long i = (long long)blockIdx.x * kStepThreads + threadIdx.x;  // b * dim + d
  if (i >= (long long)p.batch * p.dim) return;
  const long long b = i / p.dim, d = i - b * p.dim;
  const float x = p.x[b * p.xs[0] + d * p.xs[1]];
  float dt = p.dt[b * p.dts[0] + d * p.dts[1]] + (p.bias ? p.bias[d] : 0.0f);
  if (p.softplus) dt = softplus(dt);
  float* h = p.state + i * p.N;
  const float* A = p.A + d * p.N;
  const float* B = p.B + b * p.Bs[0];
  const float* C = p.C + b * p.Cs[0];
  const float dx = dt * x;
  float y = 0.0f;
  for (int n = 0; n < p.N; ++n) {
    const float hn = fmaf(fexp(dt * A[n]), h[n], dx * B[n * p.Bs[1]]);
    h[n] = hn;
    y = fmaf(C[n * p.Cs[1]], hn, y);
  }
  if (p.D) y = fmaf(p.D[d], x, y);
  if (p.z) y *= silu(p.z[b * p.zs[0] + d * p.zs[1]]);
  p.out[i] = y;
}

}  // namespace

hipError_t m1_step(const M1Step& p, hipStream_t st) {
  const long long rows = (long long)p.batch * p.dim;
  auto a16 = [](const void* q) { return ((uintptr_t)q & 15u) == 0; };
  if (p.N % 4 == 0 && a16(p.state) && a16(p.A)) {
    int Q = 1;
    while (Q < 16 && (p.N / 4) % (2 * Q) == 0) Q *= 2;
    // few rows: blocks of one wave, so that they spread over the CUs
    const int threads = rows * Q < 65536 ? 64 : kStepThreads;
    const long long blocks = (rows * Q + threads - 1) / threads;
    if (blocks <= 0 || blocks > 0x7fffffffLL) return hipErrorInvalidValue;
    const bool vb = p.Bs[1] == 1 && p.Cs[1] == 1 && p.Bs[0] % 4 == 0 && p.Cs[0] % 4 == 0 &&
                    a16(p.B) && a16(p.C);
    if (vb)
      hipLaunchKernelGGL(m1_step_vec_kernel<true>, dim3((unsigned)blocks), dim3(threads), 0, st,
                         p, Q);
    else
      hipLaunchKernelGGL(m1_step_vec_kernel<false>, dim3((unsigned)blocks), dim3(threads), 0, st,
                         p, Q);
    return hipGetLastError();
  }
  const long long blocks = (rows + kStepThreads - 1) / kStepThreads;
  if (blocks <= 0 || blocks > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(m1_step_kernel, dim3((unsigned)blocks), dim3(kStepThreads), 0, st, p);
  return hipGetLastError();
}

}  // namespace armscan
