// Deterministic column reduction of per-workgroup partial rows: out[a][c] += Σ_g part[a][g][c].
//
// The G rows are taken in S slices of up to sqrt(G) rows, and the slices' sums are added in slice order. Fixed order => bitwise
// reproducible, and the same bits in every form:
//   * on a stream that has the card to itself one launch: a workgroup takes 32 columns and 32 of the slices at a time, a thread a
//     slice of a column (its loads independent); the sums meet in LDS. As two launches the 972 rows of GPT-2's norms at 3885
//     tokens take 9.8 + 9.2 us, the 64 of a step of 256 tokens 3.9 + 4.1, beside two launches' host time;
//   * beside a second stream's work, of fewer than 1024 rows (up to 3072 tokens of a Gemma step), two launches, one row at a
//     time: a workgroup per 256 columns and slice, then one per 256 columns. Gemma-3 1B on two streams, 1024 / 1536 / 2048 / 3072
//     tokens: 22.8 / 27.3 / 29.1 / 36.1 ms a step so, 24.5 / 28.3 / 29.5 / 36.0 with one launch of 8 slices at a time. (Eight rows'
//     loads in flight give the CUs to the next kernels of both streams at once: with a layer's products at its end 1024 / 1536 / 2048
//     tokens take 23.6 / 27.7 / 31.3 so, 22.8 / 27.7 / 30.2 with one row at a time.)
//   * beside a second stream's work, of more rows, one launch of 8 slices at a time, in workgroups of 4 waves: Gemma-3 1B,
//     4096 / 6144 / 8192 tokens 42.1 / 56.2 / 65.9 ms a step so, 42.9 / 56.6 / 66.2 as two launches; GPT-2, 64 x 1024 61.1 / 61.4
//     (one launch of 32 slices, whose 16 waves rarely find room on a CU: 0.5 more); 24 layers of 1024, 8192 tokens 27.5 / 27.8.
#pragma once
#include <hip/hip_runtime.h>
#include "host_plan.h"

namespace penroz {
namespace {  // internal linkage: every including translation unit gets its own copy

struct OutPtrs {
  float* p[3];
};

// NS slices at a time
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

// whether rows beside another stream's work are summed in two launches
inline bool reduce_in_two(int G) { return G < 1024; }

// part: [A][G][C] fp32 (A <= 3); outs[a] fp32 [C] (accumulated into); shared: another stream has work for the CUs too; mid: then, if
// reduce_in_two(G), room for A·S·C floats (S = reduce_slices(G))
inline void reduce_partials_add(const float* part, int A, int G, int C, float* const* outs, hipStream_t stream,
                                bool shared = false, float* mid = nullptr) {
  OutPtrs o{};
  for (int a = 0; a < A; ++a) o.p[a] = outs[a];
  const int S = reduce_slices(G);
  const dim3 grid((C + 31) / 32, A);
  if (!shared) {
    hipLaunchKernelGGL(reduce_columns_kernel<32>, grid, dim3(1024), 0, stream, part, G, C, S, o);
  } else if (mid == nullptr) {
    hipLaunchKernelGGL(reduce_columns_kernel<8>, grid, dim3(256), 0, stream, part, G, C, S, o);
  } else {
    hipLaunchKernelGGL(reduce_slices_kernel, dim3((C + 255) / 256, S, A), dim3(256), 0, stream, part, G, C, S, mid);
    hipLaunchKernelGGL(reduce_sums_kernel, dim3((C + 255) / 256, A), dim3(256), 0, stream, mid, C, S, o);
  }
}

}  // namespace
}  // namespace penroz
