// Decode linears. A GPT block's decode step of 1 to 64 rows costs 5 launches instead of 8:
//
//   decode_ln_gemm : out = act(LN(resid) · Wᵀ + bias)          (QKV; fc + GELU)
//   decode_gemm_acc: resid += x · Wᵀ + bias                     (proj; fc2; rows_gemm.hip)
//
// The residual stream stays fp32 and is updated IN PLACE by decode_gemm_acc's epilogue, so
// the separate "residual add + LayerNorm" kernel between the GEMMs disappears: the next
// decode_ln_gemm normalises the rows it needs itself. Two choices keep that redundant
// normalisation cheap (a kernel that normalised all 64 rows in every 16-column workgroup lost at 64 rows,
// profiles/decode_fused_rows_r2.log):
//   * a decode_ln_gemm workgroup owns up to 16 ROWS × 16 to 64 columns, so it normalises only its rows;
//   * its weights are on the way meanwhile.
// Row blocks of one column tile are placed on one XCD (blockIdx % 8 picks the XCD), so the
// 4 row blocks' weight reads after the first hit that XCD's L2.
//
// MFMA: v_mfma_f32_16x16x32_bf16 with A = 16 weight rows (output columns n), B = 16 x rows
// (decode rows m): lane holds D[n = 4(lane>>4) + r][m = lane & 15], r = 0..3 — four
// consecutive outputs of one row, stored as 8 B.
#include "common.h"
#include <type_traits>
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

namespace penroz {

typedef short dl_bf16x8 __attribute__((ext_vector_type(8)));
typedef float dl_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t dl_u32x4 __attribute__((ext_vector_type(4)));

constexpr int kDlMaxSteps = 32;  // decode_ln_gemm: K <= 1024 (up to 4 quads of a row per lane)
constexpr int kDlGroup = 32;     // decode_gemm: k-steps per wave whose loads are issued together

// (row block, column tile) of a workgroup: the nrb row blocks of column tile ct share
// blockIdx % 8 (one XCD) for the full groups of 8 tiles; the tail is row-block-major.
__device__ __forceinline__ void dl_tile(int id, int nrb, int nct, int& rb, int& ct) {
  const int full = (nct / 8) * 8 * nrb;
  if (id < full) {
    const int g = 8 * nrb;
    ct = (id / g) * 8 + (id & 7);
    rb = (id % g) >> 3;
  } else {
    const int r = id - full;
    ct = (nct / 8) * 8 + r / nrb;
    rb = r % nrb;
  }
}

// Sums over the wave of R values per lane at once (R 1, 2 or 4): two values share every step of the butterfly, so R of them take
// little more than one (each by itself: 13 instructions a sum). Afterwards a lane holds the sum of value sum_of<R>(lane).
template <int R>
__device__ __forceinline__ int sum_of(int lane) {
  return R == 1 ? 0 : R == 2 ? lane >> 5 : (lane >> 5) + 2 * ((lane >> 4) & 1);
}
template <int R>
__device__ __forceinline__ float wave_sums(const float (&s)[R]) {
  static_assert(R == 1 || R == 2 || R == 4, "");
  auto over32 = [](float a, float b) {  // the lower half gets the sums of a, the upper one those of b
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  };
  auto over16 = [](float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
  };
  const float lo = over32(s[0], s[R > 1]);
  float u = over16(lo, R == 4 ? over32(s[R - 2], s[R - 1]) : lo);
  u += dpp_f32<0xB1>(u);   // quad_perm [1,0,3,2]
  u += dpp_f32<0x4E>(u);   // quad_perm [2,3,0,1]
  u += dpp_f32<0x141>(u);  // row_half_mirror
  u += dpp_f32<0x140>(u);  // row_mirror
  return u;
}
template <int R>
__device__ __forceinline__ float sum_at(float u, int i) {  // value i's, for every lane
  return R == 1 ? u : lane_f32(u, R == 2 ? 32 * i : 32 * (i & 1) + 16 * (i >> 1));
}

__device__ __forceinline__ uint2 ln_quad(const float4_t& d, float rstd, const float4_t& g, const float4_t& b) {
  return uint2{pack_bf16x2(d[0] * rstd * g[0] + b[0], d[1] * rstd * g[1] + b[1]),
               pack_bf16x2(d[2] * rstd * g[2] + b[2], d[3] * rstd * g[3] + b[3])};
}

// A wave's steps s0 .. s1 - 1 of K, its weights in registers. (With every read of x before the first product, and the steps past the
// wave's own on zeros instead of behind a branch, GPT-2's steps took 1 to 3 % longer.)
template <int SMAX>
__device__ __forceinline__ dl_f32x4 ln_products(const dl_u32x4 (&wv)[SMAX], const bf16* xl, int s0, int s1) {
  dl_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < SMAX; ++u)
    if (s0 + u < s1) {
      const dl_u32x4 xb = *reinterpret_cast<const dl_u32x4*>(xl + 32 * (s0 + u));
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dl_bf16x8, wv[u]), __builtin_bit_cast(dl_bf16x8, xb), acc, 0, 0,
                                                    0);
    }
  return acc;
}

// The end of both LayerNorm products: this wave's sums over its share of K (wave: column block cb, share kh of KS) meet those of the
// others; bias, and GELU on the bf16-rounded linear output (the unfused pair's rounding point).
template <int NB, int KS>
__device__ __forceinline__ void ln_end(dl_f32x4 acc, dl_f32x4* kred, int cb, int kh, int lane, uint2 bias_v, bool store,
                                       bf16* __restrict__ o, int act) {
  if (kh > 0) kred[((kh - 1) * NB + cb) * 64 + lane] = acc;
  __syncthreads();
  if (kh > 0 || !store) return;
#pragma unroll
  for (int p = 0; p < KS - 1; ++p) acc += kred[(p * NB + cb) * 64 + lane];
  const float bv[4] = {__uint_as_float(bias_v.x << 16), __uint_as_float(bias_v.x & 0xffff0000u), __uint_as_float(bias_v.y << 16),
                       __uint_as_float(bias_v.y & 0xffff0000u)};
  float y[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    y[r] = acc[r] + bv[r];
    if (act) y[r] = gelu_f(bf2f(from_f<bf16>(y[r])), act - 1);
  }
  *reinterpret_cast<uint2*>(o) = uint2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
}

// out = act(LN(resid) · Wᵀ + bias), 5 rows or more. A workgroup owns 4·RPW rows × 16·NB columns: the first 4 waves normalise RPW rows
// each (fp32, two passes over the row in registers) into LDS, and all its waves hold their shares of the weights in registers, asked
// for behind the residual, whose reads (L2) then come back first. JC = ceil(K / 256): quads of a row per lane.
// Bound by the chain launch, loads, sums, MFMAs, store, and from two workgroups on a CU by what one CU reads (48 KB of residual and
// 24 KB of weights per 16 columns at K = 768). So NB is the smallest, up to 4, that leaves every workgroup a CU of its own (256 of
// them; 64 x 2304 x 768 with NB 1 to 4: 6.4, 6.2, 5.0, 5.7 us). us, K 768: N 2304 at 8 / 16 / 32 / 64 rows 3.5 / 4.0 / 4.4 / 5.0,
// N 3072 4.2 / 4.5 / 4.9 / 5.6; with weights by LDS-DMA beside 4 waves that sum each row by itself, always 32 columns: 5.4 / 5.7 /
// 5.7 / 6.8 and 5.9 / 6.2 / 6.2 / 7.4. K 1024, N 4096: 4.4 / 4.6 / 5.6 / 7.2, so 6.5 / 7.2 / 7.3 / 12.0.
template <int JC, int RPW, int NB>
__global__ void __launch_bounds__(NB == 1 ? 256 : NB == 3 ? 384 : 512) decode_ln_gemm_kernel(
    const float* __restrict__ resid, const float* __restrict__ gamma, const float* __restrict__ beta, float eps,
    const bf16* __restrict__ w, const bf16* __restrict__ bias, bf16* __restrict__ out, int64_t o_rs, int M, int N, int K, int act) {
  constexpr int NW = NB == 1 ? 4 : NB == 3 ? 6 : 8, KS = NW / NB, MB = 4 * RPW, SMAX = 8 * JC / KS;
  __shared__ __attribute__((aligned(16))) bf16 xs[MB * (256 * JC + 8)];
  __shared__ __attribute__((aligned(16))) dl_f32x4 kred[(KS - 1) * NB * 64];
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int rb, ct;
  dl_tile(blockIdx.x, (M + MB - 1) / MB, (N + 16 * NB - 1) / (16 * NB), rb, ct);
  const int LDX = K + 8, steps = K / 32;  // (+16 B per row: a fragment's row reads spread over the banks)
  const int r16 = lane & 15, kq = 8 * (lane >> 4), cb = wid % NB, kh = wid / NB;
  // rows past M and quads past K are read from the last one
  float4_t r[RPW][JC], g[JC], b[JC];
  if (wid < 4) {
#pragma unroll
    for (int i = 0; i < RPW; ++i)
#pragma unroll
      for (int j = 0; j < JC; ++j)
        r[i][j] = *reinterpret_cast<const float4_t*>(resid + (size_t)min(rb * MB + wid + 4 * i, M - 1) * K +
                                                     min(4 * lane + 256 * j, K - 4));
#pragma unroll
    for (int j = 0; j < JC; ++j) {
      g[j] = *reinterpret_cast<const float4_t*>(gamma + min(4 * lane + 256 * j, K - 4));
      b[j] = *reinterpret_cast<const float4_t*>(beta + min(4 * lane + 256 * j, K - 4));
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // the loads below stay behind those above
  const int s0 = steps * kh / KS, s1 = steps * (kh + 1) / KS, nrow = (ct * NB + cb) * 16;
  const bf16* wp = w + (size_t)min(nrow + r16, N - 1) * K + kq;
  dl_u32x4 wv[SMAX];
#pragma unroll
  for (int s = 0; s < SMAX; ++s) wv[s] = *reinterpret_cast<const dl_u32x4*>(wp + 32 * min(s0 + s, steps - 1));
  const int m = rb * MB + r16, n = nrow + 4 * (lane >> 4);
  uint2 bias_v{0u, 0u};
  if (bias && kh == 0 && n < N) bias_v = *reinterpret_cast<const uint2*>(bias + n);
  __builtin_amdgcn_sched_barrier(0);
  if (wid < 4) {
    const float inv_k = 1.f / (float)K;
    const bool last = 4 * lane + 256 * (JC - 1) < K;  // the lane's last quad is one of the row
    float s[RPW], q[RPW];
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      s[i] = 0.f;
#pragma unroll
      for (int j = 0; j < JC; ++j) {
        const float v = (r[i][j][0] + r[i][j][1]) + (r[i][j][2] + r[i][j][3]);
        s[i] += j < JC - 1 || last ? v : 0.f;
      }
    }
    const float mean = wave_sums<RPW>(s) * inv_k;
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const float mi = sum_at<RPW>(mean, i);
      q[i] = 0.f;
#pragma unroll
      for (int j = 0; j < JC; ++j) {
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          r[i][j][k] -= mi;
          v += r[i][j][k] * r[i][j][k];
        }
        q[i] += j < JC - 1 || last ? v : 0.f;
      }
    }
    const float rstd = rsqrtf(wave_sums<RPW>(q) * inv_k + eps);
#pragma unroll
    for (int i = 0; i < RPW; ++i) {
      const float ri = sum_at<RPW>(rstd, i);
#pragma unroll
      for (int j = 0; j < JC; ++j)
        if (j < JC - 1 || last)
          *reinterpret_cast<uint2*>(xs + (wid + 4 * i) * LDX + 4 * lane + 256 * j) = ln_quad(r[i][j], ri, g[j], b[j]);
    }
  }
  // a barrier for LDS alone: __syncthreads would wait for the weights as well
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  const dl_f32x4 acc = ln_products<SMAX>(wv, xs + min(r16, MB - 1) * LDX + kq, s0, s1);
  ln_end<NB, KS>(acc, kred, cb, kh, lane, bias_v, n < N && m < M && r16 < MB, out + (size_t)m * o_rs + n, act);
}

// The same for up to R = 1, 2 or 4 rows: 16 columns per workgroup of 4 waves, each with 256 columns of all the rows; the waves' sums
// and squares about their own means meet in LDS (Chan's rule, as exact as two passes over the row). EMB: the residual rows are
// wte[token] + wpe[position] (the first block of a decode step, embed_fwd_kernel's arithmetic: clamped token, position min(*epos, P -
// 1)) and are written to `resid`. us at 1 / 2 / 4 rows: N 2304, K 768 2.9 / 3.1 / 3.3, where waves of their own that each normalise all
// the rows took 3.7 / 5.2 / 7.8; N 3072 3.6 / 3.7 / 4.0, so 3.9 / 5.5 / 8.0; N 4096, K 1024 3.7 / 3.8 / 3.8, so 4.7 / 6.5 / 10.6.
template <int JC, int R, bool EMB>
__global__ void __launch_bounds__(256) decode_ln_few_kernel(float* __restrict__ resid, const float* __restrict__ gamma,
                                                            const float* __restrict__ beta, float eps, const bf16* __restrict__ w,
                                                            const bf16* __restrict__ bias, bf16* __restrict__ out, int64_t o_rs,
                                                            int M, int N, int K, int act, const int64_t* __restrict__ eidx,
                                                            const bf16* __restrict__ ewte, const bf16* __restrict__ ewpe,
                                                            const int64_t* __restrict__ epos, int eV, int eP) {
  constexpr int SMAX = 2 * JC;
  __shared__ __attribute__((aligned(16))) bf16 xs[R * (256 * JC + 8)];
  __shared__ __attribute__((aligned(16))) float2 part[R][4];
  __shared__ __attribute__((aligned(16))) dl_f32x4 kred[3 * 64];
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int LDX = K + 8, steps = K / 32, c = 4 * threadIdx.x, cc = min(c, K - 4);
  const int r16 = lane & 15, kq = 8 * (lane >> 4);
  float4_t r[R];
  uint2 te[R], pe{0u, 0u};
  if constexpr (EMB) {
    const int64_t p = *epos;
    pe = *reinterpret_cast<const uint2*>(ewpe + (size_t)(p < eP ? p : eP - 1) * K + cc);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      int64_t tok = eidx[min(i, M - 1)];
      tok = tok < 0 ? 0 : tok >= eV ? eV - 1 : tok;
      te[i] = *reinterpret_cast<const uint2*>(ewte + (size_t)tok * K + cc);
    }
  } else {
#pragma unroll
    for (int i = 0; i < R; ++i) r[i] = *reinterpret_cast<const float4_t*>(resid + (size_t)min(i, M - 1) * K + cc);
  }
  const float4_t g = *reinterpret_cast<const float4_t*>(gamma + cc), b = *reinterpret_cast<const float4_t*>(beta + cc);
  __builtin_amdgcn_sched_barrier(0);
  const int s0 = steps * wid / 4, s1 = steps * (wid + 1) / 4, nrow = blockIdx.x * 16;
  const bf16* wp = w + (size_t)min(nrow + r16, N - 1) * K + kq;
  dl_u32x4 wv[SMAX];
#pragma unroll
  for (int s = 0; s < SMAX; ++s) wv[s] = *reinterpret_cast<const dl_u32x4*>(wp + 32 * min(s0 + s, steps - 1));
  const int n = nrow + 4 * (lane >> 4);
  uint2 bias_v{0u, 0u};
  if (bias && wid == 0 && n < N) bias_v = *reinterpret_cast<const uint2*>(bias + n);
  __builtin_amdgcn_sched_barrier(0);
  const bool ok = c < K;
  if constexpr (EMB) {
    auto quad = [](uint2 u) {
      return float4_t{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                      __uint_as_float(u.y & 0xffff0000u)};
    };
#pragma unroll
    for (int i = 0; i < R; ++i) {
      r[i] = quad(te[i]) + quad(pe);
      if (blockIdx.x == 0 && ok && i < M) *reinterpret_cast<float4_t*>(resid + (size_t)i * K + c) = r[i];
    }
  }
  float2 mine{0.f, 0.f};
  if (256 * wid < K) {
    const float inv_c = 1.f / (float)min(K - 256 * wid, 256);
    float s[R], q[R];
#pragma unroll
    for (int i = 0; i < R; ++i) s[i] = ok ? (r[i][0] + r[i][1]) + (r[i][2] + r[i][3]) : 0.f;
    mine.x = wave_sums<R>(s);
    const float mu = mine.x * inv_c;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const float mi = sum_at<R>(mu, i);
      float v = 0.f;
#pragma unroll
      for (int k = 0; k < 4; ++k) v += (r[i][k] - mi) * (r[i][k] - mi);
      q[i] = ok ? v : 0.f;
    }
    mine.y = wave_sums<R>(q);
  }
  if ((lane & 15) == 0) part[sum_of<R>(lane)][wid] = mine;
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if (256 * wid < K) {
    const float inv_k = 1.f / (float)K;
    const float2* pr = part[sum_of<R>(lane)];
    float2 p[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) p[x] = pr[x];
    const float mean = ((p[0].x + p[1].x) + (p[2].x + p[3].x)) * inv_k;
    float sq = 0.f;
#pragma unroll
    for (int x = 0; x < JC; ++x) {
      const float cnt = (float)min(K - 256 * x, 256), d = p[x].x / cnt - mean;
      sq += p[x].y + cnt * d * d;
    }
    const float rstd = rsqrtf(sq * inv_k + eps);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const float mi = sum_at<R>(mean, i), ri = sum_at<R>(rstd, i);
      if (ok) *reinterpret_cast<uint2*>(xs + i * LDX + c) = ln_quad(r[i] - mi, ri, g, b);
    }
  }
  __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  const dl_f32x4 acc = ln_products<SMAX>(wv, xs + min(r16, R - 1) * LDX + kq, s0, s1);
  ln_end<1, 4>(acc, kred, 0, wid, lane, bias_v, n < N && r16 < M && r16 < R, out + (size_t)r16 * o_rs + n, act);
}

// out[M, N] = x · Wᵀ (bf16) (16 rows × 16 columns per workgroup, the 4
// waves split K, partial tiles reduced through LDS; every load of a wave's k-range in flight at
// once) with a plain store, or with GATED the packed [gate; up] weight [2I, K]: a workgroup takes
// gate columns n0..n0+15 and the matching up columns I + n0.., out[m, n] = bf16(act(bf16(g)) ·
// bf16(u)) — the rounding of GEMM -> gated_act_packed. For the Gemma decode program's 17-64-row
// steps, where hipBLASLt's picks for these skinny shapes ran 36-216 workgroups (gate|up at 64
// rows: 72 workgroups, 1.6 TB/s of weights; profiles/notes_r6.md).
// RB row blocks of 16 per workgroup share each weight fragment (RB = 4 at 33-64 rows and wide N:
// the weights are read once instead of once per row block).
template <bool GATED, int RB>
__global__ void __launch_bounds__(256) decode_gemm_kernel(const bf16* __restrict__ x, int64_t x_rs,
                                                          const bf16* __restrict__ w, bf16* __restrict__ out,
                                                          int64_t o_rs, int M, int N, int K, int kind) {
  constexpr int GROUP = (GATED ? 16 : kDlGroup) / RB;
  __shared__ __attribute__((aligned(16))) dl_f32x4 red[2][RB][3 * 64];
  const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
  int rbg, ct;
  dl_tile(blockIdx.x, (M + 16 * RB - 1) / (16 * RB), N / 16, rbg, ct);
  const int steps = K / 32;
  const int s0 = steps * wid / 4, s1 = steps * (wid + 1) / 4;
  const int r16 = lane & 15, kq = 8 * (lane >> 4);
  const int n0 = ct * 16;
  const bf16* wp = w + (size_t)(n0 + r16) * K + kq;
  const bf16* up = wp + (size_t)N * K;  // GATED: the up row of the same column
  const bf16* xp[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    const int mx = (rbg * RB + r) * 16 + r16;
    xp[r] = x + (size_t)(mx < M ? mx : 0) * x_rs + kq;  // rows past M feed unstored outputs
  }
  dl_f32x4 acc0[RB], acc1[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) acc0[r] = acc1[r] = dl_f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s = s0; s < s1; s += GROUP) {
    dl_u32x4 wg[GROUP], wu[GROUP], xb[RB * GROUP];  // (flat: a 2-D array of these miscompiled)
#pragma unroll
    for (int u = 0; u < GROUP; ++u) {
      if (s + u < s1) {
        const size_t ko = (size_t)(s + u) * 32;
        wg[u] = *reinterpret_cast<const dl_u32x4*>(wp + ko);
        if constexpr (GATED) wu[u] = *reinterpret_cast<const dl_u32x4*>(up + ko);
#pragma unroll
        for (int r = 0; r < RB; ++r) xb[r * GROUP + u] = *reinterpret_cast<const dl_u32x4*>(xp[r] + ko);
      }
    }
#pragma unroll
    for (int u = 0; u < GROUP; ++u) {
      if (s + u < s1) {
#pragma unroll
        for (int r = 0; r < RB; ++r) {
          acc0[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dl_bf16x8, wg[u]),
                                                            __builtin_bit_cast(dl_bf16x8, xb[r * GROUP + u]), acc0[r], 0, 0, 0);
          if constexpr (GATED)
            acc1[r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(dl_bf16x8, wu[u]),
                                                              __builtin_bit_cast(dl_bf16x8, xb[r * GROUP + u]), acc1[r], 0, 0, 0);
        }
      }
    }
  }
  if (wid) {
#pragma unroll
    for (int r = 0; r < RB; ++r) {
      red[0][r][(wid - 1) * 64 + lane] = acc0[r];
      if constexpr (GATED) red[1][r][(wid - 1) * 64 + lane] = acc1[r];
    }
  }
  __syncthreads();
  if (wid) return;
  const int n = n0 + 4 * (lane >> 4);
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    const int m = (rbg * RB + r) * 16 + r16;
    if (m >= M) continue;
    dl_f32x4 a0 = acc0[r] + red[0][r][lane] + red[0][r][64 + lane] + red[0][r][128 + lane];
    dl_f32x4 a1 = acc1[r];
    if constexpr (GATED) a1 += red[1][r][lane] + red[1][r][64 + lane] + red[1][r][128 + lane];
    float y[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (GATED)
        y[i] = act_f(bf2f(from_f<bf16>(a0[i])), kind) * bf2f(from_f<bf16>(a1[i]));
      else
        y[i] = a0[i];
    }
    *reinterpret_cast<uint2*>(out + (size_t)m * o_rs + n) = uint2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
  }
}

// ------------------------------------------------------------------------------------------
// Decode GEMV for M <= 4 rows (batch-1..4 decode): out[M, N] = act(x · Wᵀ + bias), x either a
// bf16 matrix or — LN mode — LayerNorm(resid_in + delta + dbias) computed in the kernel (the
// residual sum also written to resid_out by workgroup 0). At these shapes a kernel's time is its
// fixed costs: launch, one memory round trip, reductions. So:
//   * one wave per workgroup, no LDS, no barrier: a half-wave (32 lanes) owns one weight row, a
//     wave 2·RP rows; lane l reads 16-B chunks l, l+32, ... of its row (512 contiguous bytes per
//     half-wave instruction) and the matching chunks of x;
//   * every load of the wave — all its weight chunks, its x (or residual / delta / bias / γ / β)
//     chunks — is issued before the first use: one round trip;
//   * LN mode normalises each row within the half-wave (fp32 two-pass on the register copy, the
//     add+LayerNorm kernel's math), rounds to bf16 (the GEMM operand's precision);
//   * products by v_dot2c_f32_bf16 (bf16 pairs into fp32), one 5-step half-wave reduction per
//     (row, x row), stores from lane 0 of each half.
// No MFMA: at M <= 4 a 16x16 MFMA tile would waste ≥ 3/4 of itself, and the VALU work is small.
typedef __bf16 dv_bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float dot8_bf16(const uint4& a, const uint4& b, float c) {
  c = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(dv_bf16x2, a.x), __builtin_bit_cast(dv_bf16x2, b.x), c, false);
  c = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(dv_bf16x2, a.y), __builtin_bit_cast(dv_bf16x2, b.y), c, false);
  c = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(dv_bf16x2, a.z), __builtin_bit_cast(dv_bf16x2, b.z), c, false);
  c = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(dv_bf16x2, a.w), __builtin_bit_cast(dv_bf16x2, b.w), c, false);
  return c;
}

// Sum over the 32 lanes of this half-wave: the butterfly over lane bits 0 to 4, without the five serial trips through
// the LDS crossbar (~100 cycles each) that __shfl_xor takes. Once a quad's lanes agree, mirroring 8 lanes reaches
// what xor 4 would, and mirroring the row what xor 8 would: the same sums in the same order.
__device__ __forceinline__ float half_sum(float v) {
  v += dpp_f32<0xB1>(v);   // quad_perm [1,0,3,2]
  v += dpp_f32<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dpp_f32<0x141>(v);  // row_half_mirror
  v += dpp_f32<0x140>(v);  // row_mirror
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float other_half(float v, int half) {  // lane ^ 32
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(half ? r[0] : r[1]);
}

// 16 bytes of weights. PAST: by a load that no cache keeps, 6.4 to 7.2 TB/s from memory where others take 5.7 to 6.3 (200 to 640 MB).
// The caller says so for weights that the 256 MB in front of the memory cannot hold from one step to the next (past_caches,
// ops/gemm.py); what they leave there is what a step finds of its other weights. Generation of 64 tokens, GPT-2 124M, one row, the head
// so: 14.95 -> 14.45 ms, but 14.94 with its layers' weights (170 MB) read so too; of 32 tokens, Gemma-3 1B, 3 rows: 34.9 -> 33.4, 33.7
// with QKV and output projections too. Weights that the caches do hold are slower so: 2 x 1024 x 1792 gated, 22 MB in all, 4 rows 5.6 ->
// 7.0 us, 6912 x 6912 24.0 -> 26.8. (Kernels of their own: a choice at run time costs one 0.3 us.)
template <bool PAST>
__device__ __forceinline__ uint4 weight16(const bf16* p) {
  if constexpr (PAST) return __builtin_bit_cast(uint4, __builtin_nontemporal_load(reinterpret_cast<const dl_u32x4*>(p)));
  else return *reinterpret_cast<const uint4*>(p);
}

// PRO: 0 — x is the bf16 operand; 1 — LN mode (GPT: fp32 residual + delta + dbias, LayerNorm)
template <int M, int PRO, int RP, int CPL, bool PAST>
__global__ void __launch_bounds__(64) decode_gemv_kernel(
    const float* __restrict__ rin, const bf16* __restrict__ delta, const float* __restrict__ dbias,
    float* __restrict__ rout, const float* __restrict__ gamma, const float* __restrict__ beta, float eps,
    const bf16* __restrict__ x, int64_t x_rs, const bf16* __restrict__ w, const bf16* __restrict__ bias,
    bf16* __restrict__ out, int64_t o_rs, int N, int K, int act, const int64_t* __restrict__ eidx = nullptr, const bf16* __restrict__ ewte = nullptr,
    const bf16* __restrict__ ewpe = nullptr, const int64_t* __restrict__ epos = nullptr, int eV = 0, int eP = 0) {
  constexpr bool LN = PRO == 1;
  const int lane = threadIdx.x, h = lane >> 5, l32 = lane & 31;
  const int nc = K / 8;  // 16-B chunks per row
  const int n0 = blockIdx.x * 2 * RP;
  auto row_of = [&](int rp) -> int { return min(n0 + 2 * rp + h, N - 1); };  // this half's rp-th weight row
  // 1. every load first, in the order of use (the vector-memory counter drains in order): the LayerNorm's operands,
  // then the weight chunks of this half's rows, whose flight covers the LayerNorm. Loads are never behind a branch on
  // a lane or behind an earlier load's use: with the residual, delta and bias of each chunk added as they came, and
  // γ, β and the bias loaded where they were needed, a LayerNorm kernel spent five memory round trips one after the
  // other (GPT-2 B = 1: 6.8 us against 3.6 for the same bytes without it).
  // Where all of that is more than 256 registers, one wave per SIMD (the estimate is the compiler's count within 15), the
  // weights come first and the LayerNorm's operands a row of x at a time (all at once / so, us: 4 rows of x, K 768,
  // N 50257 52.6 / 42.9; 3 rows, K 1024 64.1 / 44.4; but 3 rows, K 768, 245 registers, 29.7 / 36.6).
  constexpr bool EARLY = CPL * (28 + 12 * M + 5 * RP) <= 260;
  int cc[CPL];  // chunks past the row are read from its last one and count as zero
#pragma unroll
  for (int i = 0; i < CPL; ++i) cc[i] = min(l32 + 32 * i, nc - 1);
  uint4 wv[RP][CPL], xb[M][CPL];
  auto weights = [&]() {
#pragma unroll
    for (int rp = 0; rp < RP; ++rp) {
      const bf16* wr = w + (size_t)row_of(rp) * K;
#pragma unroll
      for (int i = 0; i < CPL; ++i) {
        const int c = l32 + 32 * i;
        wv[rp][i] = c < nc ? weight16<PAST>(wr + 8 * c) : uint4{0u, 0u, 0u, 0u};
      }
    }
  };
  float bias_v[RP];
#pragma unroll
  for (int rp = 0; rp < RP; ++rp) bias_v[rp] = 0.f;
  auto biases = [&]() {
    if (bias) {
#pragma unroll
      for (int rp = 0; rp < RP; ++rp) bias_v[rp] = bf2f(bias[row_of(rp)]);
    }
  };
  if constexpr (!LN) {
    biases();
    weights();
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int i = 0; i < CPL; ++i) {
        const int c = l32 + 32 * i;
        xb[m][i] = c < nc ? *reinterpret_cast<const uint4*>(x + (size_t)m * x_rs + 8 * c) : uint4{0u, 0u, 0u, 0u};
      }
  } else {
    // a chunk's values before they are added: the fp32 residual (or in embedding mode the position row's 16 bytes in
    // its first piece), then delta (the token's row)
    typedef uint32_t raw4 __attribute__((ext_vector_type(4)));
    constexpr int ME = EARLY ? M : 1;
    raw4 r4[ME][CPL][2], d4[ME][CPL];
    float4_t db4[CPL][2], gm[CPL][2], bt4[CPL][2];
    float v[M][CPL][8];
    const int epos_v = ewte ? min((int)*epos, eP - 1) : 0;
    auto load_row = [&](int m) {
      const int q = EARLY ? m : 0;
      if (ewte) {  // embedding mode: the residual row is wte[token] + wpe[position] (the first block of a decode
                   // step, embed_fwd_kernel's arithmetic: clamped token, position min(*epos, P - 1))
        int64_t tok = eidx[m];
        tok = tok < 0 ? 0 : (tok >= eV ? eV - 1 : tok);
#pragma unroll
        for (int i = 0; i < CPL; ++i) {
          d4[q][i] = *reinterpret_cast<const raw4*>(ewte + (size_t)tok * K + 8 * cc[i]);
          r4[q][i][0] = *reinterpret_cast<const raw4*>(ewpe + (size_t)epos_v * K + 8 * cc[i]);
        }
      } else {
#pragma unroll
        for (int i = 0; i < CPL; ++i) {
          const raw4* rp = reinterpret_cast<const raw4*>(rin + (size_t)m * K + 8 * cc[i]);
          r4[q][i][0] = rp[0];
          r4[q][i][1] = rp[1];
        }
        if (delta) {
#pragma unroll
          for (int i = 0; i < CPL; ++i) d4[q][i] = *reinterpret_cast<const raw4*>(delta + (size_t)m * K + 8 * cc[i]);
        }
      }
    };
    auto add_row = [&](int m) {
      const int q = EARLY ? m : 0;
#pragma unroll
      for (int i = 0; i < CPL; ++i) {
        const bool ok = l32 + 32 * i < nc;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const auto half16 = [&](const raw4& u) {
            return __uint_as_float(k & 1 ? u[k >> 1] & 0xffff0000u : u[k >> 1] << 16);
          };
          float r;
          if (ewte) {
            r = half16(d4[q][i]) + half16(r4[q][i][0]);
          } else {
            r = __uint_as_float(r4[q][i][k >> 2][k & 3]);
            if (delta) r += dbias ? half16(d4[q][i]) + db4[i][k >> 2][k & 3] : half16(d4[q][i]);
          }
          v[m][i][k] = ok ? r : 0.f;
        }
      }
    };
    auto load_dbias = [&]() {
      if (dbias) {
#pragma unroll
        for (int i = 0; i < CPL; ++i) {
          const float4_t* e = reinterpret_cast<const float4_t*>(dbias + 8 * cc[i]);
          db4[i][0] = e[0];
          db4[i][1] = e[1];
        }
      }
    };
    auto scales = [&](int i) {
      const float4_t* gp = reinterpret_cast<const float4_t*>(gamma + 8 * cc[i]);
      const float4_t* bp = reinterpret_cast<const float4_t*>(beta + 8 * cc[i]);
      gm[i][0] = gp[0];
      gm[i][1] = gp[1];
      bt4[i][0] = bp[0];
      bt4[i][1] = bp[1];
    };
    if constexpr (EARLY) {
#pragma unroll
      for (int m = 0; m < M; ++m) load_row(m);
      load_dbias();
#pragma unroll
      for (int i = 0; i < CPL; ++i) scales(i);
      biases();
      weights();
#pragma unroll
      for (int m = 0; m < M; ++m) add_row(m);
    } else {
      weights();
      load_dbias();
#pragma unroll
      for (int m = 0; m < M; ++m) {
        load_row(m);
        add_row(m);
      }
    }
    if ((delta || ewte) && rout && blockIdx.x == 0 && h == 0) {
#pragma unroll
      for (int m = 0; m < M; ++m)
#pragma unroll
        for (int i = 0; i < CPL; ++i) {
          const int c = l32 + 32 * i;
          if (c < nc) {
            float4_t* op = reinterpret_cast<float4_t*>(rout + (size_t)m * K + 8 * c);
            op[0] = float4_t{v[m][i][0], v[m][i][1], v[m][i][2], v[m][i][3]};
            op[1] = float4_t{v[m][i][4], v[m][i][5], v[m][i][6], v[m][i][7]};
          }
        }
    }
    const float inv_k = 1.f / (float)K;
    float mean[M], rstd[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < CPL; ++i)
#pragma unroll
        for (int k = 0; k < 8; ++k) s += v[m][i][k];
      mean[m] = half_sum(s) * inv_k;
    }
#pragma unroll
    for (int m = 0; m < M; ++m) {
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < CPL; ++i) {
        const bool ok = l32 + 32 * i < nc;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          const float d = v[m][i][k] - mean[m];
          ss += ok ? d * d : 0.f;
        }
      }
      rstd[m] = rsqrtf(half_sum(ss) * inv_k + eps);
    }
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
      const bool ok = l32 + 32 * i < nc;
      if constexpr (!EARLY) scales(i);
#pragma unroll
      for (int m = 0; m < M; ++m) {
        float y[8];
#pragma unroll
        for (int k = 0; k < 8; ++k)
          y[k] = ok ? (v[m][i][k] - mean[m]) * rstd[m] * gm[i][k >> 2][k & 3] + bt4[i][k >> 2][k & 3] : 0.f;
        xb[m][i] = uint4{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]), pack_bf16x2(y[4], y[5]),
                         pack_bf16x2(y[6], y[7])};
      }
    }
  }
  if constexpr (LN && !EARLY) biases();
  // 2. products and the half-wave reductions
  float acc[RP][M];
#pragma unroll
  for (int rp = 0; rp < RP; ++rp)
#pragma unroll
    for (int m = 0; m < M; ++m) {
      float a = 0.f;
#pragma unroll
      for (int i = 0; i < CPL; ++i) a = dot8_bf16(wv[rp][i], xb[m][i], a);
      acc[rp][m] = half_sum(a);
    }
  // 3. epilogue
  // a lane per output: one after the other on one lane the activations of 8 rows, 4 of x, take as long as the loads
  static_assert(RP * M <= 32, "");
  float mine = 0.f;
#pragma unroll
  for (int rp = 0; rp < RP; ++rp)
#pragma unroll
    for (int m = 0; m < M; ++m) mine = l32 == rp * M + m ? acc[rp][m] + bias_v[rp] : mine;
  const int n = n0 + 2 * (l32 / M) + h;
  if (l32 >= RP * M || n >= N) return;
  if (act) mine = gelu_f(bf2f(from_f<bf16>(mine)), act - 1);
  out[(size_t)(l32 % M) * o_rs + n] = from_f<bf16>(mine);
}

// The decode GEMV of up to 16k outputs: NW waves share the columns of RP weight rows (wave w, lane l: 16-B chunks l + 64 w, l + 64 (w +
// NW), ...), every load of a wave in flight before the first use, x first. ADD: out (fp32) += the sum, whose old value is fetched with
// the operands. At one row of x a call costs its weights' way through memory; each further row was read again by the one wave per
// weight row that there was before, so long rows (K > 4608) are shared out two to a pair of waves: half the reads of x. us before /
// now at 1, 3 and 4 rows: 1152 x 6912 5.3 / 5.2, 8.6 / 6.2, 9.9 / 6.7 (rows alone in 4 waves 6.8 at 3 rows, 4 rows in 4 waves 6.9, 8
// in 7 waves 6.3), 768 x 3072 2.8 / 2.7, 3.3 / 3.0, 3.5 / 3.2, 1152 x 1024 2.4 / 2.4, 2.8 / 2.6, 3.0 / 2.7.
template <int M, int RP, int NW, int CPL, bool ADD, bool PAST>
__global__ void __launch_bounds__(64 * NW) decode_gemv_rows_kernel(const bf16* __restrict__ x, int64_t x_rs,
                                                                   const bf16* __restrict__ w, const bf16* __restrict__ bias,
                                                                   void* __restrict__ out, int64_t o_rs, int N, int K, int act) {
  __shared__ float red[NW][RP * M];
  const int t = threadIdx.x, lane = t & 63, wid = __builtin_amdgcn_readfirstlane(t >> 6);
  const int nc = K / 8, n0 = blockIdx.x * RP;
  // thread t < RP * M: output row t % M, column n0 + t / M; the others read the last one's
  const int e = min(t, RP * M - 1), n = n0 + e / M;
  const bool mine = t < RP * M && n < N;
  const size_t o = (size_t)(e % M) * o_rs + min(n, N - 1);
  const uint16_t* bp = reinterpret_cast<const uint16_t*>(bias ? bias : x);  // (a value of x, not used, is as quick)
  uint32_t bias_v = bp[bias ? min(n, N - 1) : 0];
  float old = 0.f;
  if constexpr (ADD) old = reinterpret_cast<const float*>(out)[o];
  int cc[CPL];  // chunks past the row are read from its last one and count as zero
#pragma unroll
  for (int i = 0; i < CPL; ++i) cc[i] = min(lane + 64 * (wid + NW * i), nc - 1);
  uint4 xb[M][CPL], wv[RP][CPL];
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int i = 0; i < CPL; ++i) xb[m][i] = *reinterpret_cast<const uint4*>(x + (size_t)m * x_rs + 8 * cc[i]);
#pragma unroll
  for (int r = 0; r < RP; ++r)
#pragma unroll
    for (int i = 0; i < CPL; ++i) wv[r][i] = weight16<PAST>(w + (size_t)min(n0 + r, N - 1) * K + 8 * cc[i]);
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" : "+v"(bias_v), "+v"(old));  // asked for with the others: left to itself, each is fetched where it is needed
#pragma unroll
  for (int i = 0; i < CPL; ++i)
    if (lane + 64 * (wid + NW * i) >= nc)
#pragma unroll
      for (int m = 0; m < M; ++m) {
        xb[m][i] = uint4{0u, 0u, 0u, 0u};
        for (int r = 0; m == 0 && r < RP; ++r) wv[r][i] = uint4{0u, 0u, 0u, 0u};  // (0 · inf)
      }
  float y = bias ? __uint_as_float(bias_v << 16) : 0.f;
#pragma unroll
  for (int r = 0; r < RP; ++r)
#pragma unroll
    for (int m = 0; m < M; ++m) {
      float a = 0.f;
#pragma unroll
      for (int i = 0; i < CPL; ++i) a = dot8_bf16(wv[r][i], xb[m][i], a);
      a = half_sum(a);
      a += other_half(a, lane >> 5);
      if constexpr (NW == 1)
        y += lane == r * M + m ? a : 0.f;
      else if (lane == 0)
        red[wid][r * M + m] = a;
    }
  if constexpr (NW > 1) {
    __syncthreads();
    if (mine) {
      float a = 0.f;
#pragma unroll
      for (int i = 0; i < NW; ++i) a += red[i][t];
      y += a;
    }
  }
  if (!mine) return;
  if (act) y = gelu_f(bf2f(from_f<bf16>(y)), act - 1);
  if constexpr (ADD)
    reinterpret_cast<float*>(out)[o] = old + y;
  else
    reinterpret_cast<bf16*>(out)[o] = from_f<bf16>(y);
}

// What stands in front of a pair product: nothing, or the step between two sublayers of a Gemma block (rms_residual_kernel's math and
// rounding points): v = rms(x + a)·w1 (mode 0), x + rms(a)·w1 (1), x + a (2) or x alone (3); h = v, the product's x = rms(v)·w2. In
// mode 3 with token ids x is their rows of `table`, times `scale`.
struct PairNorm {
  const bf16 *x, *a, *w1, *w2;
  bf16* h;
  int mode;
  float eps1, eps2;
  const int64_t* tok;
  const bf16* table;
  int64_t vocab;
  float scale;
};

// Pairs of weight rows, a half-wave each, x once per workgroup in LDS (with every wave fetching it, a call of 3 rows of x
// read more of x than of weights). GATED: on the packed [gate; up] weight (N = 2I rows): half 0 takes gate row n, half 1 up row I + n,
// out[n] = act_f(bf16(g), kind) · bf16(u) (skinny_gated's rounding). Otherwise RoPE QKV: pair p of head p / (D/2), j = p % (D/2): half
// 0 row head·D + j, half 1 row + D/2, both rounded to bf16, then rotated by one position's cos / sin [D/2] for the first nrot heads
// (skinny_qkv_rope's math). A wave owns RP pairs. us before / now at 1, 3 and 4 rows, 2 x 6912 x 1152 gated: 8.0 / 7.3, 10.2 / 7.6,
// 11.2 / 7.8 (32 MB of weights; 2 pairs per wave 8.1 at 3 rows, 3 8.8, 4 8.1).
// NORM: the first M waves each make a row of x from nm, while the weights are on their way; workgroup 0 writes h. Gated, 8 waves and
// 2 pairs a wave, so that each CU repeats the rows' work at most twice, in 128 registers, so that it holds two (one with 132: 12.1 us).
// In steps of Gemma-3 1B, 3 rows: step and QKV 4.0 + 3.5 us as two kernels, 5.4 as one, step and gate|up 4.0 + 8.6, 10.9 as one.
template <int M, int RP, int CPL, int NW, bool GATED, bool NORM, bool PAST>
__global__ void __launch_bounds__(64 * NW, NORM && CPL <= 5 ? 4 : 1) decode_gemv_pair_kernel(const bf16* __restrict__ x, int64_t x_rs,
                                                                   const bf16* __restrict__ w, bf16* __restrict__ out, int64_t o_rs,
                                                                   int N, int K, int kind, int D, int nrot,
                                                                   const float* __restrict__ cosv, const float* __restrict__ sinv,
                                                                   PairNorm nm) {
  constexpr int T = 64 * NW, XN = M * 32 * CPL, XL = (XN + T - 1) / T, NV = (CPL + 1) / 2;
  static_assert(RP * M <= 32 && M <= NW, "a lane per output, a wave per row");
  __shared__ uint4 xs[XN];
  const int t = threadIdx.x, lane = t & 63, wid = __builtin_amdgcn_readfirstlane(t >> 6), h = lane >> 5, l32 = lane & 31;
  const int nc = K / 8, npair = N / 2, hd = D / 2;
  const int p0 = (blockIdx.x * NW + wid) * RP;
  uint4 wv[RP][CPL];  // chunks past a row are read from its last one and count as zero
  auto weights = [&]() {
#pragma unroll
    for (int r = 0; r < RP; ++r) {
      const int p = min(p0 + r, npair - 1), row = GATED ? p + h * npair : p / hd * D + p % hd + h * hd;
#pragma unroll
      for (int i = 0; i < CPL; ++i) wv[r][i] = weight16<PAST>(w + (size_t)row * K + 8 * min(l32 + 32 * i, nc - 1));
    }
  };
  const int p = p0 + l32 / M;  // this lane's output pair, row l32 % M of x
  const bool mine = l32 < RP * M && p < npair;
  float cs = 1.f, sn = 0.f;
  auto angles = [&]() {
    if constexpr (!GATED) {
      if (mine && p / hd < nrot) {
        cs = cosv[p % hd];
        sn = sinv[p % hd];
      }
    }
  };
  if constexpr (NORM) {
    uint4 rx[NV], ra[NV], r1[NV], r2[NV];
    if (wid < M) {
      const bf16* xr = nm.x + (size_t)wid * K;
      if (nm.tok) {
        int64_t tok = nm.tok[wid];
        tok = tok < 0 ? 0 : tok >= nm.vocab ? nm.vocab - 1 : tok;
        xr = nm.table + (size_t)tok * K;
      }
#pragma unroll
      for (int i = 0; i < NV; ++i) rx[i] = *reinterpret_cast<const uint4*>(xr + 8 * min(lane + 64 * i, nc - 1));
      if (nm.mode != 3)
#pragma unroll
        for (int i = 0; i < NV; ++i) ra[i] = *reinterpret_cast<const uint4*>(nm.a + (size_t)wid * K + 8 * min(lane + 64 * i, nc - 1));
      if (nm.mode < 2)
#pragma unroll
        for (int i = 0; i < NV; ++i) r1[i] = *reinterpret_cast<const uint4*>(nm.w1 + 8 * min(lane + 64 * i, nc - 1));
#pragma unroll
      for (int i = 0; i < NV; ++i) r2[i] = *reinterpret_cast<const uint4*>(nm.w2 + 8 * min(lane + 64 * i, nc - 1));
    }
    __builtin_amdgcn_sched_barrier(0);
    weights();
    angles();
    __builtin_amdgcn_sched_barrier(0);
    if (wid < M) {
      auto rounded = [](float f) { return bf2f(from_f<bf16>(f)); };
      float v[NV][8], xv[NV][8];
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const bool ok = lane + 64 * i < nc;
        Vec8<bf16>::load(reinterpret_cast<const bf16*>(&rx[i]), xv[i]);
        if (nm.mode != 3) Vec8<bf16>::load(reinterpret_cast<const bf16*>(&ra[i]), v[i]);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (nm.mode == 3) v[i][e] = nm.tok ? rounded(xv[i][e] * nm.scale) : xv[i][e];
          else if (nm.mode != 1) v[i][e] = rounded(xv[i][e] + v[i][e]);
          if (nm.mode < 2 && ok) ss += v[i][e] * v[i][e];
        }
      }
      if (nm.mode < 2) {
        const float r = rsqrtf(wave_sum(ss) / K + nm.eps1);
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          float w1v[8];
          Vec8<bf16>::load(reinterpret_cast<const bf16*>(&r1[i]), w1v);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float n = rounded(rounded(v[i][e] * r) * w1v[e]);
            v[i][e] = nm.mode == 0 ? n : rounded(xv[i][e] + n);
          }
        }
      }
      ss = 0.f;
#pragma unroll
      for (int i = 0; i < NV; ++i)
        if (lane + 64 * i < nc)
#pragma unroll
          for (int e = 0; e < 8; ++e) ss += v[i][e] * v[i][e];
      const float r = rsqrtf(wave_sum(ss) / K + nm.eps2);
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int j = lane + 64 * i;
        if (nm.h != nullptr && blockIdx.x == 0 && j < nc) Vec8<bf16>::store(nm.h + (size_t)wid * K + 8 * j, v[i]);
        float w2v[8];
        Vec8<bf16>::load(reinterpret_cast<const bf16*>(&r2[i]), w2v);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = j < nc ? rounded(v[i][e] * r) * w2v[e] : 0.f;
        if (j < 32 * CPL) Vec8<bf16>::store(reinterpret_cast<bf16*>(xs + wid * 32 * CPL + j), v[i]);
      }
    }
  } else {
    uint4 xt[XL];
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int e = t + T * i;
      xt[i] = *reinterpret_cast<const uint4*>(x + (size_t)min(e / (32 * CPL), M - 1) * x_rs + 8 * min(e % (32 * CPL), nc - 1));
    }
    weights();
    angles();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < XL; ++i) launder(xt[i]);  // asked for before the weights, all of them (not where a branch needs one)
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int e = t + T * i;
      if (e < XN) xs[e] = e % (32 * CPL) < nc ? xt[i] : uint4{0u, 0u, 0u, 0u};
    }
  }
  // a barrier for LDS alone: __syncthreads would wait for the weights as well
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  float acc[RP][M];
#pragma unroll
  for (int r = 0; r < RP; ++r)
#pragma unroll
    for (int m = 0; m < M; ++m) acc[r][m] = 0.f;
#pragma unroll
  for (int i = 0; i < CPL; ++i) {
    if (l32 + 32 * i >= nc)
#pragma unroll
      for (int r = 0; r < RP; ++r) wv[r][i] = uint4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const uint4 xv = xs[m * 32 * CPL + l32 + 32 * i];
#pragma unroll
      for (int r = 0; r < RP; ++r) acc[r][m] = dot8_bf16(wv[r][i], xv, acc[r][m]);
    }
  }
  float a = 0.f, b = 0.f;  // this half's row and the other's
#pragma unroll
  for (int r = 0; r < RP; ++r)
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const float v = half_sum(acc[r][m]), u = other_half(v, h);
      a = l32 == r * M + m ? v : a;
      b = l32 == r * M + m ? u : b;
    }
  if (!mine) return;
  a = bf2f(from_f<bf16>(a));
  b = bf2f(from_f<bf16>(b));
  bf16* o = out + (size_t)(l32 % M) * o_rs;
  if constexpr (GATED) {
    if (h == 0) o[p] = from_f<bf16>(act_f(a, kind) * b);
  } else {
    const float y = p / hd < nrot ? (h == 0 ? a * cs - b * sn : a * cs + b * sn) : a;
    o[p / hd * D + p % hd + h * hd] = from_f<bf16>(y);
  }
}

}  // namespace penroz

using namespace penroz;

static void dl_check_w(const torch::Tensor& w, int K, const char* who) {
  TORCH_CHECK(w.is_cuda() && w.scalar_type() == torch::kBFloat16 && w.dim() == 2 && w.is_contiguous() &&
                  w.size(1) == K && w.size(0) % 16 == 0 && reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
              who, ": bf16 contiguous 16-B aligned W [N, K], N % 16 == 0");
}

static const bf16* dl_bias(const c10::optional<torch::Tensor>& bias, int N, const char* who) {
  if (!bias.has_value() || !bias->defined()) return nullptr;
  TORCH_CHECK(bias->scalar_type() == torch::kBFloat16 && bias->is_contiguous() && bias->numel() == N &&
                  reinterpret_cast<uintptr_t>(bias->data_ptr()) % 8 == 0,
              who, ": bf16 bias [N], 8-B aligned");
  return reinterpret_cast<const bf16*>(bias->data_ptr());
}

// act(0 + bias) in every row of out: a product over no columns. The kernels clamp their loads to a row's last piece, which
// rows of no columns do not have.
static void no_columns(const c10::optional<torch::Tensor>& bias, const torch::Tensor& out, int64_t act) {
  if (!bias.has_value() || !bias->defined()) {
    out.zero_();  // (the activations' value at 0)
    return;
  }
  torch::Tensor y = bias->view({1, -1});
  out.copy_(act ? at::gelu(y.to(torch::kFloat32), act == 2 ? "tanh" : "none") : y);
}

struct LnEmb {  // the residual rows are the step's embeddings
  const int64_t* idx = nullptr;
  const bf16 *wte = nullptr, *wpe = nullptr;
  const int64_t* pos = nullptr;
  int V = 0, P = 0;
};

// K % 32 == 0, K <= 1024, N % 16 == 0, rows of out and the bias of 8-byte pieces; emb: up to 4 rows
static void ln_launch(float* resid, const float* gamma, const float* beta, float eps, const bf16* w, const bf16* bias, bf16* out,
                      int64_t o_rs, int M, int N, int K, int act, const LnEmb* emb) {
  auto stream = at::hip::getCurrentHIPStream();
  auto few = [&](auto jc, auto r, auto e) {
    constexpr int JC = decltype(jc)::value, R = decltype(r)::value;
    constexpr bool EMB = decltype(e)::value;
    const LnEmb none, &m = emb ? *emb : none;
    hipLaunchKernelGGL((decode_ln_few_kernel<JC, R, EMB>), dim3((N + 15) / 16), dim3(256), 0, stream, resid, gamma, beta, eps, w,
                       bias, out, o_rs, M, N, K, act, m.idx, m.wte, m.wpe, m.pos, m.V, m.P);
  };
  auto rows = [&](auto jc, auto rpw, auto nb) {
    constexpr int JC = decltype(jc)::value, RPW = decltype(rpw)::value, NB = decltype(nb)::value;
    const int grid = ((M + 4 * RPW - 1) / (4 * RPW)) * ((N + 16 * NB - 1) / (16 * NB));
    hipLaunchKernelGGL((decode_ln_gemm_kernel<JC, RPW, NB>), dim3(grid), dim3(NB == 1 ? 256 : NB == 3 ? 384 : 512), 0, stream, resid,
                       gamma, beta, eps, w, bias, out, o_rs, M, N, K, act);
  };
  auto typed = [&](auto jc) {
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    using Four = std::integral_constant<int, 4>;
    if (M <= 4) {
      auto by_rows = [&](auto e) {
        if (M == 1) few(jc, One{}, e);
        else if (M == 2) few(jc, Two{}, e);
        else few(jc, Four{}, e);
      };
      if (emb) by_rows(std::true_type{});
      else by_rows(std::false_type{});
      return;
    }
    if (M <= 8) return rows(jc, Two{}, One{});
    // the smallest tile that leaves each workgroup one of the 256 CUs
    const int64_t blocks = (int64_t)((M + 15) / 16) * (N / 16);
    if (blocks <= 256) rows(jc, Four{}, One{});
    else if (blocks <= 512) rows(jc, Four{}, Two{});
    else if (blocks <= 768) rows(jc, Four{}, std::integral_constant<int, 3>{});
    else rows(jc, Four{}, Four{});
  };
  if (K <= 256) typed(std::integral_constant<int, 1>{});
  else if (K <= 512) typed(std::integral_constant<int, 2>{});
  else if (K <= 768) typed(std::integral_constant<int, 3>{});
  else typed(std::integral_constant<int, 4>{});
}

// out[M, N] = act(LayerNorm(resid) · wᵀ + bias); act 0 none, 1 GELU (erf), 2 GELU (tanh).
void decode_ln_gemm(torch::Tensor resid, torch::Tensor gamma, torch::Tensor beta, double eps, torch::Tensor w,
                    c10::optional<torch::Tensor> bias, torch::Tensor out, int64_t act) {
  TORCH_CHECK(resid.is_cuda() && resid.scalar_type() == torch::kFloat32 && resid.dim() == 2 && resid.is_contiguous(),
              "decode_ln_gemm: fp32 contiguous resid [M, K]");
  const int M = resid.size(0), K = resid.size(1);
  TORCH_CHECK(M >= 1 && K % 32 == 0 && K <= 32 * kDlMaxSteps, "decode_ln_gemm: K % 32 == 0, K <= 1024");
  dl_check_w(w, K, "decode_ln_gemm");
  const int N = w.size(0);
  TORCH_CHECK(gamma.scalar_type() == torch::kFloat32 && beta.scalar_type() == torch::kFloat32 && gamma.numel() == K &&
                  beta.numel() == K && gamma.is_contiguous() && beta.is_contiguous(),
              "decode_ln_gemm: fp32 gamma / beta [K]");
  TORCH_CHECK(out.scalar_type() == torch::kBFloat16 && out.dim() == 2 && out.size(0) == M && out.size(1) == N &&
                  out.stride(1) == 1 && out.stride(0) % 4 == 0 && reinterpret_cast<uintptr_t>(out.data_ptr()) % 8 == 0,
              "decode_ln_gemm: bf16 out [M, N], rows 8-B aligned");
  TORCH_CHECK(act >= 0 && act <= 2, "decode_ln_gemm: act 0 (none), 1 (GELU erf), 2 (GELU tanh)");
  const bf16* bp = dl_bias(bias, N, "decode_ln_gemm");
  if (K == 0) return no_columns(bias, out, act);
  ln_launch(resid.data_ptr<float>(), gamma.data_ptr<float>(), beta.data_ptr<float>(), (float)eps,
            reinterpret_cast<const bf16*>(w.data_ptr()), bp, reinterpret_cast<bf16*>(out.data_ptr()), out.stride(0), M, N, K, (int)act,
            nullptr);
}

// out[M, N] = x · Wᵀ (kind < 0), or with the packed [gate; up] weight [2I, K] out[M, I] =
// act(x·Wgᵀ) ⊙ (x·Wuᵀ) (kind 0 gelu, 1 gelu_tanh, 2 silu) — decode_gemm_kernel
void decode_gemm(torch::Tensor x, torch::Tensor w, torch::Tensor out, int64_t kind) {
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == torch::kBFloat16 && x.dim() == 2 && x.stride(1) == 1 &&
                  x.stride(0) % 8 == 0 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0,
              "decode_gemm: bf16 x [M, K], rows 16-B aligned");
  const int M = x.size(0), K = x.size(1);
  TORCH_CHECK(M >= 1 && K % 32 == 0, "decode_gemm: K % 32 == 0");
  dl_check_w(w, K, "decode_gemm");
  const bool gated = kind >= 0;
  TORCH_CHECK(kind <= 2, "decode_gemm: kind -1 (plain), 0 gelu, 1 gelu_tanh, 2 silu");
  const int N = gated ? w.size(0) / 2 : w.size(0);
  TORCH_CHECK(N % 16 == 0 && (!gated || w.size(0) == 2 * N), "decode_gemm: N (gated: I) % 16 == 0");
  TORCH_CHECK(out.scalar_type() == torch::kBFloat16 && out.dim() == 2 && out.size(0) == M && out.size(1) == N &&
                  out.stride(1) == 1 && out.stride(0) % 4 == 0 && reinterpret_cast<uintptr_t>(out.data_ptr()) % 8 == 0,
              "decode_gemm: bf16 out [M, N], rows 8-B aligned");
  // 4 row blocks per workgroup once there are more than two and the columns alone give >= 256
  // workgroups (weights read once); otherwise one row block per workgroup (more workgroups)
  const int rb = (M > 32 && N / 16 >= 256) ? 4 : 1;
  const int grid = ((M + 16 * rb - 1) / (16 * rb)) * (N / 16);
  auto kern = gated ? (rb == 4 ? decode_gemm_kernel<true, 4> : decode_gemm_kernel<true, 1>)
                    : (rb == 4 ? decode_gemm_kernel<false, 4> : decode_gemm_kernel<false, 1>);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, at::hip::getCurrentHIPStream(),
                     reinterpret_cast<const bf16*>(x.data_ptr()), (int64_t)x.stride(0),
                     reinterpret_cast<const bf16*>(w.data_ptr()), reinterpret_cast<bf16*>(out.data_ptr()),
                     (int64_t)out.stride(0), M, N, K, (int)(gated ? kind : 0));
}

// decode_gemv_rows_kernel by the length of a row; M <= 4, K <= 8192. past: weight16 (of rows of more than 4608 columns; shorter ones are
// kept, what a model has of them fits the caches)
template <bool ADD>
static void gemv_rows_launch(const bf16* x, int64_t x_rs, const bf16* w, const bf16* bias, void* out, int64_t o_rs, int M, int N,
                             int K, int act, bool past) {
  auto stream = at::hip::getCurrentHIPStream();
  auto go = [&](auto mt, auto rpt, auto nwt, auto cplt) {
    constexpr int MM = decltype(mt)::value, RP = decltype(rpt)::value, NW = decltype(nwt)::value, CPL = decltype(cplt)::value;
    auto kern = decode_gemv_rows_kernel<MM, RP, NW, CPL, ADD, false>;
    if constexpr (RP == 2) {
      if (past) kern = decode_gemv_rows_kernel<MM, RP, NW, CPL, ADD, true>;
    }
    hipLaunchKernelGGL(kern, dim3((N + RP - 1) / RP), dim3(64 * NW), 0, stream, x, x_rs, w, bias, out, o_rs, N, K, act);
  };
  auto by_len = [&](auto mt) {
    using C1 = std::integral_constant<int, 1>;
    using C2 = std::integral_constant<int, 2>;
    using C3 = std::integral_constant<int, 3>;
    const int nc = (K + 7) / 8;
    if (nc <= 64) go(mt, C1{}, C1{}, C1{});
    else if (nc <= 128) go(mt, C1{}, C1{}, C2{});
    else if (nc <= 192) go(mt, C1{}, C1{}, C3{});
    else if (nc <= 384) go(mt, C1{}, C3{}, C2{});
    else if (nc <= 576) go(mt, C1{}, C3{}, C3{});
    else if (nc <= 896) go(mt, C2{}, C2{}, std::integral_constant<int, 7>{});
    else go(mt, C2{}, C2{}, std::integral_constant<int, 8>{});
  };
  switch (M) {
    case 1: by_len(std::integral_constant<int, 1>{}); break;
    case 2: by_len(std::integral_constant<int, 2>{}); break;
    case 3: by_len(std::integral_constant<int, 3>{}); break;
    default: by_len(std::integral_constant<int, 4>{});
  }
}

void gemv_add(const bf16* x, int64_t x_rs, const bf16* w, const bf16* bias, float* resid, int M, int N, int K, bool past) {
  gemv_rows_launch<true>(x, x_rs, w, bias, resid, N, M, N, K, 0, past);
}

// out[M, N] = act(x · Wᵀ + bias) for M <= 4 decode rows (decode_gemv_kernel). LN mode (x
// undefined): x = LayerNorm(resid_in + delta + dbias) with γ / β, resid_out receives the sum.
// act 0 none, 1 GELU (erf), 2 GELU (tanh). rows_per_wave 2, 4 or 8 (0: by N). past: weight16, of 16384 outputs on and of long rows.
void decode_gemv(c10::optional<torch::Tensor> x, c10::optional<torch::Tensor> rin, c10::optional<torch::Tensor> delta,
                 c10::optional<torch::Tensor> dbias, c10::optional<torch::Tensor> rout,
                 c10::optional<torch::Tensor> gamma, c10::optional<torch::Tensor> beta, double eps, torch::Tensor w,
                 c10::optional<torch::Tensor> bias, torch::Tensor out, int64_t act, int64_t rows_per_wave,
                 c10::optional<torch::Tensor> emb_idx, c10::optional<torch::Tensor> emb_wte,
                 c10::optional<torch::Tensor> emb_wpe, c10::optional<torch::Tensor> emb_pos, bool past) {
  const bool ln = !(x.has_value() && x->defined());
  const bool emb = emb_wte.has_value() && emb_wte->defined();
  const int64_t* eip = nullptr;
  const bf16 *ewp = nullptr, *epp = nullptr;
  const int64_t* eps_p = nullptr;
  int eV = 0, eP = 0;
  const int N = w.size(0), K = w.size(1);
  TORCH_CHECK(w.is_cuda() && w.scalar_type() == torch::kBFloat16 && w.dim() == 2 && w.is_contiguous() &&
                  reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0 && K % 8 == 0,
              "decode_gemv: bf16 contiguous 16-B aligned W [N, K], K % 8 == 0");
  TORCH_CHECK(K <= 256 * 32, "decode_gemv: K <= 8192");
  TORCH_CHECK(act >= 0 && act <= 2, "decode_gemv: act 0 (none), 1 (GELU erf), 2 (GELU tanh)");
  int M;
  const bf16* xp = nullptr;
  int64_t x_rs = 0;
  const float *rp = nullptr, *dbp = nullptr, *gp = nullptr, *bt = nullptr;
  const bf16* dp = nullptr;
  float* rop = nullptr;
  if (!ln) {
    TORCH_CHECK(x->scalar_type() == torch::kBFloat16 && x->dim() == 2 && x->size(1) == K && x->stride(1) == 1 &&
                    x->stride(0) % 8 == 0 && reinterpret_cast<uintptr_t>(x->data_ptr()) % 16 == 0,
                "decode_gemv: bf16 x [M, K], rows 16-B aligned");
    M = x->size(0);
    xp = reinterpret_cast<const bf16*>(x->data_ptr());
    x_rs = x->stride(0);
  } else if (emb) {  // LN mode on the step's embedding rows; resid_out receives them
    TORCH_CHECK(emb_idx.has_value() && emb_wpe.has_value() && emb_pos.has_value(), "decode_gemv: embedding mode needs idx / wpe / pos");
    TORCH_CHECK(emb_idx->is_cuda() && emb_idx->scalar_type() == torch::kInt64 && emb_idx->is_contiguous(),
                "decode_gemv: int64 token ids");
    for (const torch::Tensor* t : {&*emb_wte, &*emb_wpe})
      TORCH_CHECK(t->scalar_type() == torch::kBFloat16 && t->dim() == 2 && t->is_contiguous() && t->size(1) == K && t->size(0) > 0 &&
                      reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0, "decode_gemv: bf16 contiguous wte / wpe [*, K]");
    TORCH_CHECK(emb_pos->is_cuda() && emb_pos->scalar_type() == torch::kInt64 && emb_pos->numel() == 1, "decode_gemv: int64 pos [1]");
    TORCH_CHECK(K <= 1024, "decode_gemv: LN mode needs K <= 1024");
    TORCH_CHECK(gamma.has_value() && beta.has_value() && gamma->scalar_type() == torch::kFloat32 &&
                    beta->scalar_type() == torch::kFloat32 && gamma->numel() == K && beta->numel() == K &&
                    gamma->is_contiguous() && beta->is_contiguous(), "decode_gemv: fp32 gamma / beta [K]");
    M = emb_idx->numel();
    TORCH_CHECK(rout.has_value() && rout->defined() && rout->scalar_type() == torch::kFloat32 && rout->is_contiguous() &&
                    rout->numel() == (int64_t)M * K, "decode_gemv: fp32 resid_out [M, K] for the embedding rows");
    rop = rout->data_ptr<float>();
    gp = gamma->data_ptr<float>();
    bt = beta->data_ptr<float>();
    eip = emb_idx->data_ptr<int64_t>();
    ewp = reinterpret_cast<const bf16*>(emb_wte->data_ptr());
    epp = reinterpret_cast<const bf16*>(emb_wpe->data_ptr());
    eps_p = emb_pos->data_ptr<int64_t>();
    eV = (int)emb_wte->size(0);
    eP = (int)emb_wpe->size(0);
  } else {
    TORCH_CHECK(rin.has_value() && rin->defined() && rin->scalar_type() == torch::kFloat32 && rin->dim() == 2 &&
                    rin->is_contiguous() && rin->size(1) == K, "decode_gemv: fp32 contiguous resid_in [M, K]");
    TORCH_CHECK(K <= 1024, "decode_gemv: LN mode needs K <= 1024");
    TORCH_CHECK(gamma.has_value() && beta.has_value() && gamma->scalar_type() == torch::kFloat32 &&
                    beta->scalar_type() == torch::kFloat32 && gamma->numel() == K && beta->numel() == K &&
                    gamma->is_contiguous() && beta->is_contiguous(), "decode_gemv: fp32 gamma / beta [K]");
    M = rin->size(0);
    rp = rin->data_ptr<float>();
    gp = gamma->data_ptr<float>();
    bt = beta->data_ptr<float>();
    if (delta.has_value() && delta->defined()) {
      TORCH_CHECK(delta->scalar_type() == torch::kBFloat16 && delta->is_contiguous() && delta->numel() == (int64_t)M * K,
                  "decode_gemv: bf16 contiguous delta [M, K]");
      TORCH_CHECK(rout.has_value() && rout->defined() && rout->scalar_type() == torch::kFloat32 &&
                      rout->is_contiguous() && rout->numel() == (int64_t)M * K && rout->data_ptr() != rin->data_ptr(),
                  "decode_gemv: fp32 resid_out [M, K] (not aliasing resid_in) with a delta");
      dp = reinterpret_cast<const bf16*>(delta->data_ptr());
      rop = rout->data_ptr<float>();
      if (dbias.has_value() && dbias->defined()) {
        TORCH_CHECK(dbias->scalar_type() == torch::kFloat32 && dbias->is_contiguous() && dbias->numel() == K,
                    "decode_gemv: fp32 dbias [K]");
        dbp = dbias->data_ptr<float>();
      }
    }
  }
  TORCH_CHECK(M >= 1 && M <= 4, "decode_gemv: 1..4 rows");
  TORCH_CHECK(out.scalar_type() == torch::kBFloat16 && out.dim() == 2 && out.size(0) == M && out.size(1) == N &&
                  out.stride(1) == 1, "decode_gemv: bf16 out [M, N]");
  const bf16* bp = nullptr;
  if (bias.has_value() && bias->defined()) {
    TORCH_CHECK(bias->scalar_type() == torch::kBFloat16 && bias->is_contiguous() && bias->numel() == N,
                "decode_gemv: bf16 bias [N]");
    bp = reinterpret_cast<const bf16*>(bias->data_ptr());
  }
  if (K == 0) return no_columns(bias, out, act);
  static const int rpw_env = [] {
    const char* e = std::getenv("PENROZ_DECODE_GEMV_RPW");
    return e ? std::atoi(e) : 0;
  }();
  // a LayerNorm product of whole tiles: one workgroup normalises for 16 columns (decode_ln_few_kernel). The vocabulary's many columns
  // stay with the waves below (50304 x 768, 77 MB, one row, in steps of GPT-2 124M: 14.3 us through the caches, which hold part of it, 16.2
  // past them)
  if (ln && !dp && rows_per_wave <= 0 && rpw_env <= 0 && K % 32 == 0 && N % 16 == 0 && N < 16384 && out.stride(0) % 4 == 0 &&
      reinterpret_cast<uintptr_t>(out.data_ptr()) % 8 == 0 && reinterpret_cast<uintptr_t>(bp) % 8 == 0) {
    const LnEmb e{eip, ewp, epp, eps_p, eV, eP};
    ln_launch(emb ? rop : const_cast<float*>(rp), gp, bt, (float)eps, reinterpret_cast<const bf16*>(w.data_ptr()), bp,
              reinterpret_cast<bf16*>(out.data_ptr()), out.stride(0), M, N, K, (int)act, emb ? &e : nullptr);
    return;
  }
  if (!ln && rows_per_wave <= 0 && N < 16384)
    return gemv_rows_launch<false>(xp, x_rs, reinterpret_cast<const bf16*>(w.data_ptr()), bp, out.data_ptr(), out.stride(0), M, N, K,
                                   (int)act, past);
  const int cpl = (K / 8 + 31) / 32;
  int rpw = (int)rows_per_wave;
  // by shape: the vocabulary projection wants fewer, longer-lived waves (8 rows); behind a LayerNorm 4 rows, since every
  // wave reads and normalises the whole operand again (2 / 4 / 8 rows, us: K 768, N 2304, one row of x 4.8 / 4.2 / 4.3,
  // four 10.5 / 9.0 / 8.8; K 1024, N 4096 6.7 / 5.3 / 4.9 and 13.8 / 12.1 / 12.0; K 512, N 512 3.1 / 3.2 / 3.3).
  // PENROZ_DECODE_GEMV_RPW forces 2 / 4 / 8 there below 16k rows (A/B).
  if (rpw <= 0 && rpw_env > 0 && N < 16384) rpw = rpw_env;
  if (rpw <= 0) rpw = N >= 16384 ? 8 : 4;
  TORCH_CHECK(rpw == 2 || rpw == 4 || rpw == 8, "decode_gemv: rows_per_wave 2, 4 or 8");
  const int RPv = rpw / 2;
  const dim3 grid((N + rpw - 1) / rpw);
  auto stream = at::hip::getCurrentHIPStream();
  auto wp = reinterpret_cast<const bf16*>(w.data_ptr());
  auto op = reinterpret_cast<bf16*>(out.data_ptr());
  const int64_t o_rs = out.stride(0);
  auto launch = [&](auto mt, auto lnt, auto rpt, auto cplt) {
    constexpr int MM = decltype(mt)::value, RR = decltype(rpt)::value, CC = decltype(cplt)::value;
    constexpr int LL = decltype(lnt)::value ? 1 : 0;
    auto kern = decode_gemv_kernel<MM, LL, RR, CC, false>;
    if constexpr (RR == 4) {
      if (past) kern = decode_gemv_kernel<MM, LL, RR, CC, true>;
    }
    hipLaunchKernelGGL(kern, grid, dim3(64), 0, stream, rp, dp, dbp, rop, gp, bt,
                       (float)eps, xp, x_rs, wp, bp, op, o_rs, N, K, (int)act, eip, ewp, epp, eps_p, eV, eP);
  };
  auto by_cpl = [&](auto mt, auto lnt, auto rpt) {
    using I = std::integral_constant<int, 0>;
    (void)sizeof(I);
    if (cpl <= 1) launch(mt, lnt, rpt, std::integral_constant<int, 1>{});
    else if (cpl <= 2) launch(mt, lnt, rpt, std::integral_constant<int, 2>{});
    else if (cpl <= 3) launch(mt, lnt, rpt, std::integral_constant<int, 3>{});
    else if (cpl <= 4) launch(mt, lnt, rpt, std::integral_constant<int, 4>{});
    else if (cpl <= 5) launch(mt, lnt, rpt, std::integral_constant<int, 5>{});
    else if (cpl <= 7) launch(mt, lnt, rpt, std::integral_constant<int, 7>{});
    else if (cpl <= 12) launch(mt, lnt, rpt, std::integral_constant<int, 12>{});
    else if (cpl <= 16) launch(mt, lnt, rpt, std::integral_constant<int, 16>{});
    else if (cpl <= 25) launch(mt, lnt, rpt, std::integral_constant<int, 25>{});
    else launch(mt, lnt, rpt, std::integral_constant<int, 32>{});
  };
  auto by_rp = [&](auto mt, auto lnt) {
    if (RPv == 1) by_cpl(mt, lnt, std::integral_constant<int, 1>{});
    else if (RPv == 2) by_cpl(mt, lnt, std::integral_constant<int, 2>{});
    else by_cpl(mt, lnt, std::integral_constant<int, 4>{});
  };
  auto by_ln = [&](auto mt) {
    if (ln) {
      TORCH_CHECK(cpl <= 4, "decode_gemv: LN mode needs K <= 1024");
      auto by_chunks = [&](auto rpt) {  // K <= 1024
        if (cpl <= 1) launch(mt, std::true_type{}, rpt, std::integral_constant<int, 1>{});
        else if (cpl <= 2) launch(mt, std::true_type{}, rpt, std::integral_constant<int, 2>{});
        else if (cpl <= 3) launch(mt, std::true_type{}, rpt, std::integral_constant<int, 3>{});
        else launch(mt, std::true_type{}, rpt, std::integral_constant<int, 4>{});
      };
      if (RPv == 1) by_chunks(std::integral_constant<int, 1>{});
      else if (RPv == 2) by_chunks(std::integral_constant<int, 2>{});
      else by_chunks(std::integral_constant<int, 4>{});
    } else {
      by_rp(mt, std::false_type{});
    }
  };
  switch (M) {
    case 1: by_ln(std::integral_constant<int, 1>{}); break;
    case 2: by_ln(std::integral_constant<int, 2>{}); break;
    case 3: by_ln(std::integral_constant<int, 3>{}); break;
    default: by_ln(std::integral_constant<int, 4>{});
  }
}

// Paired-row decode GEMV for 1..4 rows (decode_gemv_pair_kernel):
//   mode 1 (gated): out[M, I] = act_f(x·Wgᵀ, kind) ⊙ (x·Wuᵀ), w = [Wg; Wu] [2I, K];
//   mode 2 (RoPE QKV): out[M, (H + 2Hkv)·D] = rope(x · Wᵀ) for the first nrot heads, cos / sin [D/2].
// x is given, or nm makes it. past: weight16, of gated weights.
static void gemv_pair_launch(const bf16* xp, int64_t x_rs, const PairNorm* nm, int M, const torch::Tensor& w, const torch::Tensor& out,
                             int64_t mode, int64_t kind, int64_t D, int64_t nrot, const c10::optional<torch::Tensor>& cosv,
                             const c10::optional<torch::Tensor>& sinv, int64_t pairs_per_wave, bool past, const char* who) {
  const int N = w.size(0), K = w.size(1);
  TORCH_CHECK(mode == 1 || mode == 2, who, ": mode 1 (gated) or 2 (RoPE)");
  TORCH_CHECK(w.is_cuda() && w.scalar_type() == torch::kBFloat16 && w.dim() == 2 && w.is_contiguous() &&
                  reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0 && K % 8 == 0 && N % 2 == 0,
              who, ": bf16 contiguous 16-B aligned W [N, K], K % 8 == 0, N even");
  TORCH_CHECK(M >= 1 && M <= 4, who, ": 1..4 rows");
  const int cpl = (K / 8 + 31) / 32;
  TORCH_CHECK(cpl <= 7, who, ": K <= 1792");
  const int Nout = mode == 1 ? N / 2 : N;
  TORCH_CHECK(out.scalar_type() == torch::kBFloat16 && out.dim() == 2 && out.size(0) == M && out.size(1) == Nout &&
                  out.stride(1) == 1, who, ": bf16 out [M, N/2] (gated) or [M, N] (RoPE)");
  const float *cp = nullptr, *sp = nullptr;
  if (mode == 1) {
    TORCH_CHECK(kind >= 0 && kind <= 2, who, ": kind 0 gelu, 1 gelu_tanh, 2 silu");
  } else if (mode == 2) {
    TORCH_CHECK(D >= 2 && D % 2 == 0 && N % D == 0 && nrot >= 0 && nrot <= N / D, who, ": RoPE geometry");
    TORCH_CHECK(cosv.has_value() && sinv.has_value() && cosv->is_cuda() && sinv->is_cuda() &&
                    cosv->scalar_type() == torch::kFloat32 && sinv->scalar_type() == torch::kFloat32 &&
                    cosv->numel() >= D / 2 && sinv->numel() >= D / 2 && cosv->is_contiguous() && sinv->is_contiguous(),
                who, ": fp32 cos / sin [D/2]");
    cp = cosv->data_ptr<float>();
    sp = sinv->data_ptr<float>();
  }
  const int ppw = pairs_per_wave <= 0 ? 1 : (int)pairs_per_wave;
  TORCH_CHECK(ppw == 1 || ppw == 2 || ppw == 4, who, ": pairs_per_wave 1, 2 or 4");
  if (K == 0) {  // (as in no_columns; both forms of nothing are 0)
    out.zero_();
    return;
  }
  auto stream = at::hip::getCurrentHIPStream();
  auto wp = reinterpret_cast<const bf16*>(w.data_ptr());
  auto op = reinterpret_cast<bf16*>(out.data_ptr());
  const int64_t o_rs = out.stride(0);
  auto launch = [&](auto mt, auto rpt, auto cplt, auto et, auto nt) {
    constexpr int MM = decltype(mt)::value, RR = decltype(rpt)::value, CC = decltype(cplt)::value;
    constexpr bool GATED = decltype(et)::value, NORM = decltype(nt)::value;
    constexpr int NW = NORM && GATED ? 8 : 4;
    const dim3 grid((N / 2 + NW * RR - 1) / (NW * RR));
    auto kern = decode_gemv_pair_kernel<MM, RR, CC, NW, GATED, NORM, false>;
    if constexpr (GATED && (NORM || RR == 1)) {
      if (past) kern = decode_gemv_pair_kernel<MM, RR, CC, NW, GATED, NORM, true>;
    }
    hipLaunchKernelGGL(kern, grid, dim3(64 * NW), 0, stream, xp, x_rs, wp, op, o_rs,
                       N, K, (int)kind, mode == 1 ? 2 : (int)D, (int)nrot, cp, sp, nm ? *nm : PairNorm{});
  };
  auto by_cpl = [&](auto mt, auto rpt, auto et, auto nt) {
    if (cpl <= 3) launch(mt, rpt, std::integral_constant<int, 3>{}, et, nt);
    else if (cpl <= 4) launch(mt, rpt, std::integral_constant<int, 4>{}, et, nt);
    else if (cpl <= 5) launch(mt, rpt, std::integral_constant<int, 5>{}, et, nt);
    else launch(mt, rpt, std::integral_constant<int, 7>{}, et, nt);
  };
  auto by_mode = [&](auto mt) {
    using C1 = std::integral_constant<int, 1>;
    using C2 = std::integral_constant<int, 2>;
    auto by_rp = [&](auto et) {
      if (nm != nullptr) {
        if constexpr (decltype(et)::value) by_cpl(mt, C2{}, et, std::true_type{});
        else by_cpl(mt, C1{}, et, std::true_type{});
      }
      else if (ppw == 1) by_cpl(mt, C1{}, et, std::false_type{});
      else if (ppw == 2) by_cpl(mt, C2{}, et, std::false_type{});
      else by_cpl(mt, std::integral_constant<int, 4>{}, et, std::false_type{});
    };
    if (mode == 1) by_rp(std::true_type{});
    else by_rp(std::false_type{});
  };
  switch (M) {
    case 1: by_mode(std::integral_constant<int, 1>{}); break;
    case 2: by_mode(std::integral_constant<int, 2>{}); break;
    case 3: by_mode(std::integral_constant<int, 3>{}); break;
    default: by_mode(std::integral_constant<int, 4>{});
  }
}

void decode_gemv_pair(torch::Tensor x, torch::Tensor w, torch::Tensor out, int64_t mode, int64_t kind, int64_t D,
                      int64_t nrot, c10::optional<torch::Tensor> cosv, c10::optional<torch::Tensor> sinv,
                      int64_t pairs_per_wave, bool past) {
  TORCH_CHECK(w.dim() == 2 && x.scalar_type() == torch::kBFloat16 && x.dim() == 2 && x.size(1) == w.size(1) && x.stride(1) == 1 &&
                  x.stride(0) % 8 == 0 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0,
              "decode_gemv_pair: bf16 x [M, K], rows 16-B aligned");
  gemv_pair_launch(reinterpret_cast<const bf16*>(x.data_ptr()), x.stride(0), nullptr, (int)x.size(0), w, out, mode, kind, D, nrot, cosv,
                   sinv, pairs_per_wave, past, "decode_gemv_pair");
}

// decode_gemv_pair of x' = rms(v)·w2 with v of `step` (PairNorm's modes 0 to 3); h [M, K] receives v (optional in mode 3 without
// tokens, where it is x)
void decode_norm_pair(c10::optional<torch::Tensor> x, c10::optional<torch::Tensor> a, c10::optional<torch::Tensor> w1, torch::Tensor w2,
                      int64_t step, double eps1, double eps2, c10::optional<torch::Tensor> h, torch::Tensor w, torch::Tensor out,
                      int64_t mode, int64_t kind, int64_t D, int64_t nrot, c10::optional<torch::Tensor> cosv,
                      c10::optional<torch::Tensor> sinv, c10::optional<torch::Tensor> tok, c10::optional<torch::Tensor> table,
                      double scale, bool past) {
  const char* who = "decode_norm_pair";
  TORCH_CHECK(w.dim() == 2 && w.size(1) > 0 && step >= 0 && step <= 3, who, ": W [N, K], step 0 to 3");
  const int64_t K = w.size(1);
  auto given = [](const c10::optional<torch::Tensor>& t) { return t.has_value() && t->defined(); };
  const bool emb = given(tok);
  TORCH_CHECK(!emb || (step == 3 && given(table) && given(h)), who, ": tokens with step 3, a table and h");
  TORCH_CHECK(emb != given(x) && given(a) == (step != 3) && (step >= 2 || given(w1)), who, ": operands of the step");
  PairNorm nm{};
  int64_t M;
  if (emb) {
    TORCH_CHECK(tok->is_cuda() && tok->scalar_type() == torch::kInt64 && tok->is_contiguous(), who, ": int64 tokens");
    M = tok->numel();
  } else {
    TORCH_CHECK(x->dim() == 2, who, ": x [M, K]");
    M = x->size(0);
  }
  auto rows = [&](const torch::Tensor& t, int64_t n) {
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kBFloat16 && t.is_contiguous() && t.numel() == n * K &&
                    reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0, who, ": bf16 contiguous rows of K values, 16-B aligned");
    return reinterpret_cast<bf16*>(t.data_ptr());
  };
  if (given(x)) nm.x = rows(*x, M);
  if (given(a)) nm.a = rows(*a, M);
  if (step < 2) nm.w1 = rows(*w1, 1);
  nm.w2 = rows(w2, 1);
  if (given(h)) {
    nm.h = rows(*h, M);
    TORCH_CHECK(nm.h != nm.x && nm.h != nm.a, who, ": h apart from x and a (other workgroups still read them)");
  }
  TORCH_CHECK(step == 3 || nm.h != nullptr, who, ": h");
  nm.mode = (int)step;
  nm.eps1 = (float)eps1;
  nm.eps2 = (float)eps2;
  if (emb) {
    TORCH_CHECK(table->dim() == 2 && table->size(0) > 0, who, ": table [V, K]");
    nm.tok = tok->data_ptr<int64_t>();
    nm.vocab = table->size(0);
    nm.table = rows(*table, nm.vocab);
    nm.scale = (float)scale;
  }
  gemv_pair_launch(nullptr, 0, &nm, (int)M, w, out, mode, kind, D, nrot, cosv, sinv, 0, past, who);
}
