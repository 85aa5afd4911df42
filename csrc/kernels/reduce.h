// Deterministic column reduction of per-workgroup partial rows: out[a][c] += Σ_g part[a][g][c].
//
// The G rows are taken in S slices of up to sqrt(G) rows, and the slices' sums are added in slice order. Fixed order => bitwise
// reproducible, and the same bits in both forms:
//   * on a stream that has the card to itself one launch: a workgroup takes 32 columns and 32 of the slices at a time, a thread a
//     slice of a column (its loads independent); the sums meet in LDS. As two launches the 972 rows of GPT-2's norms at 3885
//     tokens take 9.8 + 9.2 us, the 64 of a step of 256 tokens 3.9 + 4.1, beside two launches' host time;
//   * beside a second stream's work two launches, one row at a time: a workgroup per 256 columns and slice, then one per 256
//     columns. Gemma-3 1B on two streams, 1024 / 1536 / 2048 tokens: 22.5 / 26.9 / 29.7 ms a step so, 23.7 / 27.2 / 31.0 with one
//     launch whose workgroups walk 8 slices at a time (C / 32 of them: every load waits behind the other stream's), 23.6 / 27.4 /
//     31.2 as two launches with eight rows' loads in flight (whose CUs the streams' products and AdamW then want at once).
//     GPT-2, 64 x 1024 tokens: level (63.4 ms as two launches, 63.2 as one of 8 slices at a time, 63.7 of 32).
#pragma once
#include <hip/hip_runtime.h>
#include "host_plan.h"

namespace penroz {
namespace {  // internal linkage: every including translation unit gets its own copy

struct OutPtrs {
  float* p[3];
};

constexpr int kReduceSlices = 32;

__global__ void __launch_bounds__(32 * kReduceSlices) reduce_columns_kernel(const float* __restrict__ part, int G, int C, int S,
                                                                            OutPtrs outs) {
  __shared__ float sums[kReduceSlices][32];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int c = blockIdx.x * 32 + tx, a = blockIdx.y;
  const int per = (G + S - 1) / S;
  const float* p = part + (size_t)a * G * C + c;
  float acc = 0.f;
  for (int s0 = 0; s0 < S; s0 += kReduceSlices) {
    const int s = s0 + ty, g1 = s < S && c < C ? min(G, (s + 1) * per) : 0;
    float v = 0.f;
#pragma unroll 8
    for (int g = s * per; g < g1; ++g) v += p[(size_t)g * C];
    sums[ty][tx] = v;
    __syncthreads();
    if (ty == 0)
      for (int j = 0; j < min(kReduceSlices, S - s0); ++j) acc += sums[j][tx];
    __syncthreads();
  }
  if (ty == 0 && c < C) outs.p[a][c] += acc;
}

__global__ void __launch_bounds__(256) reduce_slices_kernel(const float* __restrict__ part, int G, int C, int S,
                                                            float* __restrict__ mid) {
  const int c = blockIdx.x * 256 + threadIdx.x, s = blockIdx.y, a = blockIdx.z;
  if (c >= C) return;
  const int per = (G + S - 1) / S, g1 = min(G, (s + 1) * per);
  const float* p = part + (size_t)a * G * C + c;
  float v = 0.f;
  for (int g = s * per; g < g1; ++g) v += p[(size_t)g * C];
  mid[((size_t)a * S + s) * C + c] = v;
}

__global__ void __launch_bounds__(256) reduce_sums_kernel(const float* __restrict__ mid, int C, int S, OutPtrs outs) {
  const int c = blockIdx.x * 256 + threadIdx.x, a = blockIdx.y;
  if (c >= C) return;
  float acc = 0.f;
  for (int s = 0; s < S; ++s) acc += mid[((size_t)a * S + s) * C + c];
  outs.p[a][c] += acc;
}

// part: [A][G][C] fp32 (A <= 3); outs[a] fp32 [C] (accumulated into); mid: null, or room for A·S·C floats where another stream
// has work for the CUs too (S = reduce_slices(G))
inline void reduce_partials_add(const float* part, int A, int G, int C, float* const* outs, hipStream_t stream,
                                float* mid = nullptr) {
  OutPtrs o{};
  for (int a = 0; a < A; ++a) o.p[a] = outs[a];
  const int S = reduce_slices(G);
  if (mid == nullptr) {
    hipLaunchKernelGGL(reduce_columns_kernel, dim3((C + 31) / 32, A), dim3(32 * kReduceSlices), 0, stream, part, G, C, S, o);
    return;
  }
  hipLaunchKernelGGL(reduce_slices_kernel, dim3((C + 255) / 256, S, A), dim3(256), 0, stream, part, G, C, S, mid);
  hipLaunchKernelGGL(reduce_sums_kernel, dim3((C + 255) / 256, A), dim3(256), 0, stream, mid, C, S, o);
}

}  // namespace
}  // namespace penroz
