// Deterministic column reduction of per-workgroup partial rows: out[a][c] += Σ_g part[a][g][c].
//
// One launch: a workgroup takes 32 columns and NS of the S slices of the rows at a time, a thread a slice of a column (up to
// sqrt(G) rows, their loads independent); the slices' sums meet in LDS and are added in slice order. Fixed order => bitwise
// reproducible. As two launches (slices, then their sums) the 972 rows of GPT-2's norms at 3885 tokens took 9.8 + 9.2 us, the 64
// of a step of 256 tokens 3.9 + 4.1, beside two launches' host time. NS = 32 where the launch has the card to itself; 8, in workgroups
// of 4 waves, beside a second stream's work, whose CUs rarely have room for 16 (GPT-2, 64 x 1024 tokens: 63.4 ms a step as two
// launches, 63.7 with 32, 63.2 with 8).
#pragma once
#include <hip/hip_runtime.h>
#include "host_plan.h"

namespace penroz {
namespace {  // internal linkage: every including translation unit gets its own copy

struct OutPtrs {
  float* p[3];
};

template <int NS>
__global__ void __launch_bounds__(32 * NS) reduce_columns_kernel(const float* __restrict__ part, int G, int C, int S, OutPtrs outs) {
  __shared__ float sums[NS][32];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int c = blockIdx.x * 32 + tx, a = blockIdx.y;
  const int per = (G + S - 1) / S;
  const float* p = part + (size_t)a * G * C + c;
  float acc = 0.f;
  for (int s0 = 0; s0 < S; s0 += NS) {
    const int s = s0 + ty, g1 = s < S && c < C ? min(G, (s + 1) * per) : 0;
    float v = 0.f;
#pragma unroll 8
    for (int g = s * per; g < g1; ++g) v += p[(size_t)g * C];
    sums[ty][tx] = v;
    __syncthreads();
    if (ty == 0)
      for (int j = 0; j < min(NS, S - s0); ++j) acc += sums[j][tx];
    __syncthreads();
  }
  if (ty == 0 && c < C) outs.p[a][c] += acc;
}

// part: [A][G][C] fp32 (A <= 3); outs[a] fp32 [C] (accumulated into); shared: another stream has work for the CUs too.
inline void reduce_partials_add(const float* part, int A, int G, int C, float* const* outs, hipStream_t stream,
                                bool shared = false) {
  OutPtrs o{};
  for (int a = 0; a < A; ++a) o.p[a] = outs[a];
  const dim3 grid((C + 31) / 32, A);
  if (shared) hipLaunchKernelGGL(reduce_columns_kernel<8>, grid, dim3(256), 0, stream, part, G, C, reduce_slices(G), o);
  else hipLaunchKernelGGL(reduce_columns_kernel<32>, grid, dim3(1024), 0, stream, part, G, C, reduce_slices(G), o);
}

}  // namespace
}  // namespace penroz
