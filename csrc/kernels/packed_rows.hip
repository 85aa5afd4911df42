// Row kernels of the packed decoder step (sequences of unequal length laid end to end, no padding):
// embedding gather, residual add of a grouped RMS norm, causal convolution over time, and the
// convolution's per-sequence state. The residual stream and every statistic are fp32; T (bf16 or
// float) is the type of the sublayer outputs read here and of the sublayer inputs written here.
//
//   row_norm_add — one workgroup per row:
//       y     = the sublayer's output row, or the weighted sum of its `top` expert rows
//       x    += grouped_rms_norm(y) · nw            (skipped without y; x starts as the embedding row
//                                                    when token ids are given)
//       h     = x + conv(x)                         (decode form, one new token per sequence: the
//                                                    earlier inputs come from the state, which the
//                                                    same threads then shift)
//   conv_rows / conv_state — the convolution of many new tokens per sequence: earlier rows of the
//       same sequence from x, older ones from the state; the state moves on in a launch of its own
//       (conv_rows of other workgroups still read the old one).
//   norm_conv — row_norm_add and conv_rows of many new tokens in one pass, for norm groups that a wave holds.
//   row_norm — grouped RMS norm of selected rows (the final norm).
//   residual_norm — the step between two sublayers of a pre-norm block, one workgroup per row:
//       x  = embedding row + position row, or x + the sublayer's output: one row, `coef` times the sum of
//            two rows (each RMS-normed with its weight when it has one), or the weighted sum of `top`
//            expert rows and a shared expert's row
//       h  = rms_norm(x) · nw
// A state row k of a sequence whose last token sits at position p holds the input at position
// p - (taps - 2) + k; positions before 0 count as zero, so a reused slot needs no clearing.
#include "common.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

namespace penroz {

constexpr int kPrThreads = 256;
constexpr int kMaxTaps = 16;

// per-group 1/rms of the C values in LDS: the block sums group after group (fixed order)
__device__ __forceinline__ void group_rstd(const float* ys, int C, int groups, float eps, float* red, float* rstd) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, gs = C / groups;
  for (int g = 0; g < groups; ++g) {
    float ss = 0.f;
    for (int i = t; i < gs; i += kPrThreads) {
      const float v = ys[g * gs + i];
      ss = fmaf(v, v, ss);
    }
    ss = wave_sum(ss);
    if (lane == 0) red[g * 4 + w] = ss;
  }
  __syncthreads();
  for (int g = t; g < groups; g += kPrThreads) {
    const float s = (red[g * 4] + red[g * 4 + 1]) + (red[g * 4 + 2] + red[g * 4 + 3]);
    rstd[g] = 1.f / sqrtf(s / (float)gs + eps);
  }
  __syncthreads();
}

template <typename T>
__global__ void __launch_bounds__(kPrThreads) row_norm_add_kernel(
    const int64_t* __restrict__ tok, const T* __restrict__ table, int64_t vocab, const float* __restrict__ x_in,
    float* __restrict__ x_out, const T* __restrict__ y, const float* __restrict__ pw, int top,
    const float* __restrict__ nw, int groups, float eps, const float* __restrict__ cw, int taps,
    float* __restrict__ state, const int* __restrict__ slot, int* __restrict__ pos, int advance, T* __restrict__ h,
    int C) {
  extern __shared__ float lds[];
  float* ys = lds;                 // C
  float* red = ys + C;             // 4 · groups
  float* rstd = red + 4 * groups;  // groups
  const int row = blockIdx.x, t = threadIdx.x;
  int p = 0, sl = 0;
  if (cw != nullptr || advance) {
    p = pos[row] + advance;
    sl = slot[row];
    if (advance) {
      __syncthreads();
      if (t == 0) pos[row] = p;
    }
  }
  if (y != nullptr) {
    for (int c = t; c < C; c += kPrThreads) {
      float v;
      if (pw != nullptr) {
        v = 0.f;
        for (int k = 0; k < top; ++k)
          v = fmaf(pw[(size_t)row * top + k], to_f<T>(y[((size_t)row * top + k) * C + c]), v);
      } else {
        v = to_f<T>(y[(size_t)row * C + c]);
      }
      ys[c] = v;
    }
    __syncthreads();
    group_rstd(ys, C, groups, eps, red, rstd);
  }
  const int gs = C / groups;
  const T* erow = nullptr;
  if (tok != nullptr) {
    int64_t id = tok[row];
    PZ_DEVICE_CHECK(id >= 0 && id < vocab);
    id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
    erow = table + (size_t)id * C;
  }
  float* st = state != nullptr ? state + (size_t)sl * (taps - 1) * C : nullptr;
  for (int c = t; c < C; c += kPrThreads) {
    float x = erow != nullptr ? to_f<T>(erow[c]) : x_in[(size_t)row * C + c];
    if (y != nullptr) x = fmaf(ys[c] * rstd[c / gs], nw[c], x);
    if (x_out != nullptr) x_out[(size_t)row * C + c] = x;
    if (h != nullptr) {
      float a = x;
      if (cw != nullptr) {
        a = fmaf(cw[(size_t)(taps - 1) * C + c], x, a);
        for (int k = 0; k + 1 < taps; ++k) {
          const float s = st[(size_t)k * C + c];
          if (p - (taps - 1) + k >= 0) a = fmaf(cw[(size_t)k * C + c], s, a);
          if (k > 0) st[(size_t)(k - 1) * C + c] = s;
        }
        if (taps > 1) st[(size_t)(taps - 2) * C + c] = x;
      }
      h[(size_t)row * C + c] = from_f<T>(a);
    }
  }
}

template <typename T>
__device__ __forceinline__ float4_t load4(const T* p) {
  if constexpr (sizeof(T) == 4) {
    return *reinterpret_cast<const float4_t*>(p);
  } else {
    const uint2 u = *reinterpret_cast<const uint2*>(p);
    return float4_t{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                    __uint_as_float(u.y & 0xffff0000u)};
  }
}
template <typename T>
__device__ __forceinline__ void put4(T* p, float4_t v) {
  if constexpr (sizeof(T) == 4) *reinterpret_cast<float4_t*>(p) = v;
  else *reinterpret_cast<uint2*>(p) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

// V values as they lie in memory: a load that nothing waits for before the values are converted
template <typename T, int V>
struct alignas(sizeof(T) * V) Piece {
  T v[V];
};
template <int V, typename T>
__device__ __forceinline__ Piece<T, V> piece(const T* p) {
  return *reinterpret_cast<const Piece<T, V>*>(p);
}

// The same row with one 4-channel vector per thread (C <= 4096, parts of a multiple of 4): everything the
// row needs is loaded, and the state's share of the convolution summed, before the norm's barrier. As in residual_norm_kernel the
// loads are issued before any is waited for, the expert rows KT at a time, the state's 3; KT and CONV are
// template arguments for the registers that the simpler forms save (plain rows would lose 9 % to them; with the convolution, KT 8
// leaves one workgroup of 1024 threads per CU: 512 x 4096, 6 experts, one tap 14.4 us, KT 4 12.6). Rows of 2048, one load waited
// for at a time / here, us: 64 rows of 6 experts with the convolution 6.1 / 5.2, 8192 of 6 experts 69 / 59 (5.3 TB/s), 8192 plain
// 33.4 / 32.5; 2000 rows of 1024, 4 experts 8.6 / 7.9.
template <typename T, int KT, bool CONV>
__global__ void __launch_bounds__(1024) row_norm_add4_kernel(
    const int64_t* __restrict__ tok, const T* __restrict__ table, int64_t vocab, const float* __restrict__ x_in,
    float* __restrict__ x_out, const T* __restrict__ y, const float* __restrict__ pw, int top,
    const float* __restrict__ nw, int groups, float eps, const float* __restrict__ cw, int taps,
    float* __restrict__ state, const int* __restrict__ slot, int* __restrict__ pos, int advance, T* __restrict__ h,
    int C) {
  __shared__ float ss[1024];
  __shared__ float rstd[1024];
  const int row = blockIdx.x, t = threadIdx.x, c = 4 * t;
  const bool in = c < C;
  int p = 0, sl = 0;
  if (CONV || advance) {
    p = pos[row] + advance;
    sl = slot[row];
    if (advance) {
      __syncthreads();
      if (t == 0) pos[row] = p;
    }
  }
  float4_t x = {0.f, 0.f, 0.f, 0.f}, v = x, hist = x, wn = x, wl = x;
  float* st = state != nullptr ? state + (size_t)sl * (taps - 1) * C + c : nullptr;
  if (in) {
    if (tok != nullptr) {
      int64_t id = tok[row];
      PZ_DEVICE_CHECK(id >= 0 && id < vocab);
      id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
      x = load4<T>(table + (size_t)id * C + c);
    } else {
      x = load4<float>(x_in + (size_t)row * C + c);
    }
    if (y != nullptr) wn = load4<float>(nw + c);
    const bool past = CONV && taps > 1;
    float4_t sk[3], wk[3];
    auto load_past = [&](int k0) {
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const int k = k0 + j + 1 < taps ? k0 + j : taps - 2;
        sk[j] = load4<float>(st + (size_t)k * C);
        wk[j] = load4<float>(cw + (size_t)k * C + c);
      }
    };
    if (CONV) wl = load4<float>(cw + (size_t)(taps - 1) * C + c);
    if constexpr (KT > 0) {
      const T* first = y + (size_t)row * top * C + c;
      for (int k0 = 0; k0 < top; k0 += KT) {
        Piece<T, 4> r[KT];
        float wr[KT];
#pragma unroll
        for (int k = 0; k < KT; ++k) {
          const int kk = k0 + k < top ? k0 + k : top - 1;
          wr[k] = pw[(size_t)row * top + kk];
          r[k] = piece<4>(first + (size_t)kk * C);
        }
        if (k0 == 0 && past) load_past(0);
#pragma unroll
        for (int k = 0; k < KT; ++k) {
          const float4_t yk = load4<T>(r[k].v);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float f = fmaf(wr[k], yk[i], v[i]);
            v[i] = k0 + k < top ? f : v[i];  // a select: behind a branch its loads would wait there
          }
        }
      }
    } else {
      Piece<T, 4> r = {};
      if (y != nullptr && pw == nullptr) r = piece<4>(y + (size_t)row * C + c);
      if (past) load_past(0);
      v = load4<T>(r.v);
    }
    for (int k0 = 0; past && k0 + 1 < taps; k0 += 3) {
      if (k0 > 0) load_past(k0);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const int k = k0 + j;
        const bool seen = k + 1 < taps && p - (taps - 1) + k >= 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float f = fmaf(wk[j][i], sk[j][i], hist[i]);
          hist[i] = seen ? f : hist[i];
        }
        if (k > 0 && k + 1 < taps) put4<float>(st + (size_t)(k - 1) * C, sk[j]);
      }
    }
  }
  if (y != nullptr) {
    ss[t] = fmaf(v[0], v[0], fmaf(v[1], v[1], fmaf(v[2], v[2], v[3] * v[3])));
    __syncthreads();
    const int lane = t & 63, gv = C / groups / 4;
    for (int g = t >> 6; g < groups; g += blockDim.x >> 6) {
      float s = 0.f;
      for (int i = lane; i < gv; i += 64) s += ss[g * gv + i];
      s = wave_sum(s);
      if (lane == 0) rstd[g] = 1.f / sqrtf(s / (float)(4 * gv) + eps);
    }
    __syncthreads();
    if (in) {
      const float r = rstd[t / gv];
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = fmaf(v[i] * r, wn[i], x[i]);
    }
  }
  if (!in) return;
  if (x_out != nullptr) put4<float>(x_out + (size_t)row * C + c, x);
  if (h != nullptr) {
    float4_t a = x;
    if (CONV) {
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = fmaf(wl[i], x[i], a[i]) + hist[i];
      if (taps > 1) put4<float>(st + (size_t)(taps - 2) * C, x);
    }
    put4<T>(h + (size_t)row * C + c, a);
  }
}

template <typename T>
__global__ void __launch_bounds__(kPrThreads) row_norm_kernel(const float* __restrict__ x, const int* __restrict__ rows,
                                                              const float* __restrict__ w, int groups, float eps,
                                                              T* __restrict__ out, int C) {
  extern __shared__ float lds[];
  float* ys = lds;
  float* red = ys + C;
  float* rstd = red + 4 * groups;
  const int t = threadIdx.x;
  const size_t row = rows != nullptr ? rows[blockIdx.x] : blockIdx.x;
  for (int c = t; c < C; c += kPrThreads) ys[c] = x[row * C + c];
  __syncthreads();
  group_rstd(ys, C, groups, eps, red, rstd);
  const int gs = C / groups;
  for (int c = t; c < C; c += kPrThreads) out[(size_t)blockIdx.x * C + c] = from_f<T>(ys[c] * rstd[c / gs] * w[c]);
}

// V channels per thread; blockIdx.x: row group of 4 rows, blockIdx.y: channel block
template <typename T, int V>
__global__ void __launch_bounds__(kPrThreads) conv_rows_kernel(const float* __restrict__ x, const float* __restrict__ cw,
                                                               int taps, const float* __restrict__ state,
                                                               const int* __restrict__ slot,
                                                               const int* __restrict__ pos,
                                                               const int* __restrict__ first, T* __restrict__ h, int N,
                                                               int C) {
  const int c0 = (blockIdx.y * 64 + (threadIdx.x & 63)) * V;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= N || c0 >= C) return;
  const int p = pos[row], f = first[row];
  const float* st = state + (size_t)slot[row] * (taps - 1) * C;
  float a[V];
#pragma unroll
  for (int i = 0; i < V; ++i) a[i] = x[(size_t)row * C + c0 + i];
#pragma unroll
  for (int i = 0; i < V; ++i) a[i] = fmaf(cw[(size_t)(taps - 1) * C + c0 + i], a[i], a[i]);
  for (int j = 1; j < taps; ++j) {  // the input j positions back
    if (p - j < 0) break;
    // rows of this step first; before them the state, whose last row is the position before `first`
    const float* src = row - j >= f ? x + (size_t)(row - j) * C : st + (size_t)(taps - 1 + (row - j - f)) * C;
    const float* wj = cw + (size_t)(taps - 1 - j) * C;
#pragma unroll
    for (int i = 0; i < V; ++i) a[i] = fmaf(wj[c0 + i], src[c0 + i], a[i]);
  }
#pragma unroll
  for (int i = 0; i < V; ++i) h[(size_t)row * C + c0 + i] = from_f<T>(a[i]);
}

// x_out = x + grouped_rms_norm(y)·nw and h = x_out + conv(x_out) of many new tokens per sequence, in one pass.
// A wave holds one norm group of 256·Q channels (4 per lane and quarter), so a row's mean square is a wave reduction,
// and goes down `span` rows four at a time, the next four's loads in flight, with the last three rows of x_out in
// registers for the convolution; the three rows before its span it computes again. x_out is another buffer than x,
// whose rows the neighbour before still reads.
// Bound by memory: x and y are read and x_out and h written once (the halo adds 3 / span to the reads). With the
// state's launch, against norm and convolution one after the other: 8192 rows of 2048, 4 groups, 56 -> 38 us; 16384
// 105 -> 91; 1024 16.3 -> 13.0 (called alone over and over; between the other kernels of a prompt, 8192 rows, it takes
// 42 us, the state's launch 5). (With the weighted sum of 6 expert rows instead of y: 90 -> 91, so not here.)
constexpr int kNcTaps = 4;
template <typename T> struct Raw4 { using type = uint2; };
template <> struct Raw4<float> { using type = float4_t; };
template <typename T>
__device__ __forceinline__ float4_t raw4(typename Raw4<T>::type u) {
  if constexpr (sizeof(T) == 4) return u;
  else return float4_t{__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                       __uint_as_float(u.y & 0xffff0000u)};
}

template <int Q> constexpr int norm_conv_blocks() { return Q == 1 ? 4 : 2; }  // per CU

template <typename T, int Q>
__global__ void __launch_bounds__(kPrThreads, norm_conv_blocks<Q>()) norm_conv_kernel(
    const float* __restrict__ x, float* __restrict__ x_out, const T* __restrict__ y, const float* __restrict__ nw,
    int groups, float eps, const float* __restrict__ cw, int taps, const float* __restrict__ state,
    const int* __restrict__ slot, const int* __restrict__ pos, const int* __restrict__ first, T* __restrict__ h, int N,
    int C, int span) {
  using R = typename Raw4<T>::type;
  const int lane = threadIdx.x & 63, g = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (g >= groups) return;
  const int r0 = blockIdx.x * span, r1 = min(r0 + span, N), c = g * 256 * Q + 4 * lane;
  float4_t wn[Q], wc[kNcTaps][Q];  // wc[j]: of the input j positions back
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    wn[q] = load4<float>(nw + c + 256 * q);
#pragma unroll
    for (int j = 0; j < kNcTaps; ++j)
      wc[j][q] = j < taps ? load4<float>(cw + (size_t)(taps - 1 - j) * C + c + 256 * q) : float4_t{0.f, 0.f, 0.f, 0.f};
  }
  float4_t xr[4][Q];
  R yr[4][Q];
  auto load = [&](int row) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const size_t rr = (size_t)min(max(row + i, 0), N - 1);
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        xr[i][q] = load4<float>(x + rr * C + c + 256 * q);
        yr[i][q] = *reinterpret_cast<const R*>(y + rr * C + c + 256 * q);
      }
    }
  };
  float4_t before[3][Q];  // x_out one, two, three rows before this four's first
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int q = 0; q < Q; ++q) before[j][q] = float4_t{0.f, 0.f, 0.f, 0.f};
  load(r0 - 3);
  for (int row = r0 - 3; row < r1; row += 4) {
    float4_t xn[4][Q], v[4][Q];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        xn[i][q] = xr[i][q];
        v[i][q] = raw4<T>(yr[i][q]);
      }
    if (row + 4 < r1) load(row + 4);
    float ss[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ss[i] = 0.f;
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int k = 0; k < 4; ++k) ss[i] = fmaf(v[i][q][k], v[i][q][k], ss[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) ss[i] = wave_sum(ss[i]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float r = 1.f / sqrtf(ss[i] / (float)(256 * Q) + eps);
#pragma unroll
      for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int k = 0; k < 4; ++k) xn[i][q][k] = fmaf(v[i][q][k] * r, wn[q][k], xn[i][q][k]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int rr = row + i;
      if (rr < r0 || rr >= r1) continue;
      const int p = pos[rr], back = rr - first[rr];  // rows of the sequence before this one in the step
      const float* st = state + (size_t)slot[rr] * (taps - 1) * C;
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        float4_t a;
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k] = fmaf(wc[0][q][k], xn[i][q][k], xn[i][q][k]);
#pragma unroll
        for (int j = 1; j < kNcTaps; ++j) {
          if (j >= taps || p < j) break;
          float4_t u = i >= j ? xn[i >= j ? i - j : 0][q] : before[i >= j ? 0 : j - i - 1][q];
          if (back < j) u = load4<float>(st + (size_t)(taps - 1 + back - j) * C + c + 256 * q);
#pragma unroll
          for (int k = 0; k < 4; ++k) a[k] = fmaf(wc[j][q][k], u[k], a[k]);
        }
        put4<float>(x_out + (size_t)rr * C + c + 256 * q, xn[i][q]);
        put4<T>(h + (size_t)rr * C + c + 256 * q, a);
      }
    }
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int q = 0; q < Q; ++q) before[j][q] = xn[3 - j][q];
  }
}

__global__ void __launch_bounds__(kPrThreads) conv_state_kernel(const float* __restrict__ x, int taps,
                                                                float* __restrict__ state, const int* __restrict__ cu,
                                                                const int* __restrict__ seq_slot, int C) {
  const int s = blockIdx.x, c = blockIdx.y * kPrThreads + threadIdx.x;
  if (c >= C) return;
  const int r0 = cu[s], n = cu[s + 1] - r0;
  float* st = state + (size_t)seq_slot[s] * (taps - 1) * C + c;
  // ascending k reads entries k + n >= k + 1: each old entry is read before it is overwritten
  for (int k = 0; k + 1 < taps; ++k) {
    const int i = n - (taps - 1) + k;  // the step's row that lands in entry k
    st[(size_t)k * C] = i >= 0 ? x[(size_t)(r0 + i) * C + c] : st[(size_t)(k + n) * C];
  }
}

template <typename T>
struct ResidualArgs {
  const int64_t* tok;    // embedding rows start x (with the position rows, when there are any)
  const T *table, *ptable;
  int64_t vocab, npos;
  const float* x_in;
  float* x_out;
  const T *ya, *yb;      // the sublayer's output rows; with pw, ya holds `top` expert rows per token
  const float *wa, *wb;  // norm weights of ya / yb
  float coef, yeps;
  const float* pw;       // [N, pws]: weights of the expert rows, then the shared row's
  int top, pws;
  const T* ys;
  const float* nw;
  float eps;
  int* pos;
  int advance;
  T* h;
  int C;
};

template <typename T, int V>
__device__ __forceinline__ void load_v(const T* p, float (&v)[V]) {
  if constexpr (V == 4) {
    const float4_t a = load4<T>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = a[i];
  } else {
    v[0] = to_f<T>(p[0]);
  }
}
template <typename T, int V>
__device__ __forceinline__ void put_v(T* p, const float (&v)[V]) {
  if constexpr (V == 4) put4<T>(p, float4_t{v[0], v[1], v[2], v[3]});
  else p[0] = from_f<T>(v[0]);
}

// sums of two values over the block (up to 16 waves), in wave order
__device__ __forceinline__ float2 block_sum2(float a, float b, float2* red) {
  a = wave_sum(a);
  b = wave_sum(b);
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if ((threadIdx.x & 63) == 0) red[w] = float2{a, b};
  __syncthreads();
  float2 s = red[0];
  for (int i = 1; i < nw; ++i) {
    s.x += red[i].x;
    s.y += red[i].y;
  }
  return s;
}

// V channels per thread and pass, I passes: blockDim.x · V · I >= C. A decode step's few rows are bound by the chain of memory trips,
// so every load that does not follow from another is issued before the first is waited for: the norm weights ahead of the sums
// that they scale, the expert rows up to KM at a time. Rows of 2048, one load waited for at a time / here, us: 16 rows of 6 experts and a shared one
// 4.2 / 3.8, 64 of them 4.9 / 4.0, 8192 of them 78 / 64 (4.9 TB/s); 16 of two normed outputs 3.8 / 3.5, 4096 of them 26 / 24. One or two
// experts' rows are not read as four (one expert, 512 x 2048: 6.4 us, here 5.9). KM 4 for fp32 rows of more than 2048 values, whose
// 1024 threads are the only workgroup of a CU with the registers of KM 8 (two normed outputs, 4096 x 4096: 92 us, here 68).
template <typename T, int V, int I, int KM>
__global__ void __launch_bounds__(1024) residual_norm_kernel(ResidualArgs<T> a) {
  __shared__ float2 red[2][16];
  const int row = blockIdx.x, t = threadIdx.x, C = a.C;
  const size_t base = (size_t)row * C;
  int p = 0;
  if (a.advance || a.ptable != nullptr) {
    p = a.pos[row] + a.advance;
    if (a.advance) {
      __syncthreads();
      if (t == 0) a.pos[row] = p;
    }
  }
  const T *erow = nullptr, *prow = nullptr;
  if (a.tok != nullptr) {
    int64_t id = a.tok[row];
    PZ_DEVICE_CHECK(id >= 0 && id < a.vocab);
    id = id < 0 ? 0 : (id >= a.vocab ? a.vocab - 1 : id);
    erow = a.table + (size_t)id * C;
    if (a.ptable != nullptr) {
      PZ_DEVICE_CHECK(p >= 0 && p < a.npos);
      prow = a.ptable + (size_t)(p < 0 ? 0 : (p >= a.npos ? a.npos - 1 : p)) * C;
    }
  }
  float x[I][V], ya[I][V], yb[I][V], wa[I][V], wb[I][V], nw[I][V];
  float sa = 0.f, sb = 0.f;
#pragma unroll
  for (int i = 0; i < I; ++i) {
    const int c = (i * blockDim.x + t) * V, cc = c < C ? c : C - V;
    if (erow != nullptr) {
      load_v<T, V>(erow + cc, x[i]);
      if (prow != nullptr) {
        float q[V];
        load_v<T, V>(prow + cc, q);
#pragma unroll
        for (int j = 0; j < V; ++j) x[i][j] += q[j];
      }
    } else {
      load_v<float, V>(a.x_in + base + cc, x[i]);
    }
    if (a.wa != nullptr) load_v<float, V>(a.wa + cc, wa[i]);
    if (a.wb != nullptr) load_v<float, V>(a.wb + cc, wb[i]);
    if (I == 1 && a.nw != nullptr) load_v<float, V>(a.nw + cc, nw[i]);
    if (a.ya != nullptr) {
      // a null pointer's place is taken by the first row of ya, which is read anyway; its values are not used then
      const T* first = a.ya + (size_t)row * (a.pw != nullptr ? a.top : 1) * C + cc;
      const Piece<T, V> rb = piece<V>(a.yb != nullptr ? a.yb + base + cc : first);
      if (a.pw != nullptr) {
        const Piece<T, V> rs = piece<V>(a.ys != nullptr ? a.ys + base + cc : first);
        const float* w = a.pw + (size_t)row * a.pws;
#pragma unroll
        for (int j = 0; j < V; ++j) ya[i][j] = 0.f;
        const float ws = w[a.ys != nullptr ? a.top : 0];
        auto add = [&](float wk, const Piece<T, V>& r, bool there) {  // a select: behind a branch its loads would wait there
#pragma unroll
          for (int j = 0; j < V; ++j) {
            const float s = fmaf(wk, to_f<T>(r.v[j]), ya[i][j]);
            ya[i][j] = there ? s : ya[i][j];
          }
        };
        auto rows = [&](auto kt) {
          constexpr int KT = decltype(kt)::value;
          for (int k0 = 0; k0 < a.top; k0 += KT) {
            Piece<T, V> r[KT];
            float wk[KT];
#pragma unroll
            for (int k = 0; k < KT; ++k) {
              const int kk = k0 + k < a.top ? k0 + k : a.top - 1;
              wk[k] = w[kk];
              r[k] = piece<V>(first + (size_t)kk * C);
            }
#pragma unroll
            for (int k = 0; k < KT; ++k) add(wk[k], r[k], k0 + k < a.top);
          }
        };
        if (a.top == 1) rows(std::integral_constant<int, 1>{});
        else if (a.top == 2) rows(std::integral_constant<int, 2>{});
        else if (KM == 4 || a.top <= 4) rows(std::integral_constant<int, 4>{});
        else rows(std::integral_constant<int, 8>{});
        add(ws, rs, a.ys != nullptr);
      } else {
        load_v<T, V>(first, ya[i]);
      }
#pragma unroll
      for (int j = 0; j < V; ++j) yb[i][j] = to_f<T>(rb.v[j]);
    }
    if (c >= C) {
#pragma unroll
      for (int j = 0; j < V; ++j) x[i][j] = ya[i][j] = yb[i][j] = 0.f;
    } else if (a.ya != nullptr) {
#pragma unroll
      for (int j = 0; j < V; ++j) {
        sa = fmaf(ya[i][j], ya[i][j], sa);
        if (a.yb != nullptr) sb = fmaf(yb[i][j], yb[i][j], sb);
      }
    }
  }
  if (a.ya != nullptr) {
    float ra = 1.f, rb = 1.f;
    if (a.wa != nullptr || a.wb != nullptr) {
      const float2 s = block_sum2(sa, sb, red[0]);
      if (a.wa != nullptr) ra = 1.f / sqrtf(s.x / (float)C + a.yeps);
      if (a.wb != nullptr) rb = 1.f / sqrtf(s.y / (float)C + a.yeps);
    }
#pragma unroll
    for (int i = 0; i < I; ++i) {
      const int c = (i * blockDim.x + t) * V;
      if (c >= C) continue;
      float v[V];
#pragma unroll
      for (int j = 0; j < V; ++j) v[j] = ya[i][j] * ra;
      if (a.wa != nullptr) {
#pragma unroll
        for (int j = 0; j < V; ++j) v[j] *= wa[i][j];
      }
      if (a.yb != nullptr) {
#pragma unroll
        for (int j = 0; j < V; ++j) v[j] = fmaf(yb[i][j] * rb, a.wb != nullptr ? wb[i][j] : 1.f, v[j]);
      }
#pragma unroll
      for (int j = 0; j < V; ++j) x[i][j] = fmaf(a.coef, v[j], x[i][j]);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < I; ++i) {
    const int c = (i * blockDim.x + t) * V;
    if (c >= C) continue;
    if (a.x_out != nullptr) put_v<float, V>(a.x_out + base + c, x[i]);
#pragma unroll
    for (int j = 0; j < V; ++j) ss = fmaf(x[i][j], x[i][j], ss);
  }
  if (a.h == nullptr) return;
  const float r = 1.f / sqrtf(block_sum2(ss, 0.f, red[1]).x / (float)C + a.eps);
#pragma unroll
  for (int i = 0; i < I; ++i) {
    const int c = (i * blockDim.x + t) * V;
    if (c >= C) continue;
    if (I > 1) load_v<float, V>(a.nw + c, nw[i]);  // several passes have no registers for it before
#pragma unroll
    for (int j = 0; j < V; ++j) nw[i][j] *= x[i][j] * r;
    put_v<T, V>(a.h + base + c, nw[i]);
  }
}

}  // namespace penroz

using namespace penroz;

#define PR_CHECK_DEV(t) TORCH_CHECK((t).is_cuda() && (t).is_contiguous(), #t " must be a contiguous GPU tensor")

template <typename F>
static void pr_dispatch(at::ScalarType dt, F&& f) {
  if (dt == at::kBFloat16) f((bf16*)nullptr);
  else if (dt == at::kFloat) f((float*)nullptr);
  else TORCH_CHECK(false, "packed row kernels take bfloat16 or float32");
}

// y: [N, C], or [N·top, C] with pw [N, top]. With cw (fp32 [taps, C]) the rows are one new token of
// N different sequences. advance: pos (int32 [N]) is incremented first.
void row_norm_add(c10::optional<torch::Tensor> tok, c10::optional<torch::Tensor> table,
                  c10::optional<torch::Tensor> x_in, c10::optional<torch::Tensor> x_out,
                  c10::optional<torch::Tensor> y, c10::optional<torch::Tensor> pw, c10::optional<torch::Tensor> nw,
                  int64_t groups, double eps, c10::optional<torch::Tensor> cw, c10::optional<torch::Tensor> state,
                  c10::optional<torch::Tensor> slot, c10::optional<torch::Tensor> pos, bool advance,
                  c10::optional<torch::Tensor> h) {
  TORCH_CHECK(tok.has_value() != x_in.has_value(), "row_norm_add: token ids or x_in");
  TORCH_CHECK(x_out.has_value() || h.has_value(), "row_norm_add: nothing to write");
  int64_t N, C, vocab = 0;
  at::ScalarType dt = at::kFloat;
  if (tok.has_value()) {
    PR_CHECK_DEV(*tok);
    TORCH_CHECK(table.has_value() && tok->scalar_type() == at::kLong, "row_norm_add: int64 ids and their table");
    PR_CHECK_DEV(*table);
    N = tok->numel();
    C = table->size(1);
    vocab = table->size(0);
    dt = table->scalar_type();
  } else {
    PR_CHECK_DEV(*x_in);
    TORCH_CHECK(x_in->dim() == 2 && x_in->scalar_type() == at::kFloat, "row_norm_add: x_in is fp32 [N, C]");
    N = x_in->size(0);
    C = x_in->size(1);
  }
  if (y.has_value()) dt = y->scalar_type();
  if (h.has_value()) {
    PR_CHECK_DEV(*h);
    TORCH_CHECK((!y.has_value() && !tok.has_value()) || h->scalar_type() == dt, "row_norm_add: h dtype");
    dt = h->scalar_type();
    TORCH_CHECK(h->numel() == N * C, "row_norm_add: h is [N, C]");
  }
  if (x_out.has_value()) {
    PR_CHECK_DEV(*x_out);
    TORCH_CHECK(x_out->scalar_type() == at::kFloat && x_out->numel() == N * C, "row_norm_add: x_out is fp32 [N, C]");
  }
  int64_t top = 1;
  if (y.has_value()) {
    PR_CHECK_DEV(*y);
    TORCH_CHECK(nw.has_value() && nw->is_contiguous() && nw->scalar_type() == at::kFloat && nw->numel() == C,
                "row_norm_add: fp32 norm weight [C]");
    TORCH_CHECK(groups >= 1 && C % groups == 0 && groups <= 1024, "row_norm_add: groups");
    if (pw.has_value()) {
      PR_CHECK_DEV(*pw);
      TORCH_CHECK(pw->scalar_type() == at::kFloat && pw->dim() == 2 && pw->size(0) == N, "row_norm_add: pw [N, top]");
      top = pw->size(1);
    }
    TORCH_CHECK(y->numel() == N * top * C, "row_norm_add: y rows");
  } else {
    groups = 1;
  }
  int64_t taps = 1;
  if (cw.has_value()) {
    PR_CHECK_DEV(*cw);
    taps = cw->size(0);
    TORCH_CHECK(cw->scalar_type() == at::kFloat && cw->numel() == taps * C && h.has_value() && taps <= kMaxTaps,
                "row_norm_add: fp32 taps [taps, C] and an output");
    TORCH_CHECK(state.has_value() && state->is_contiguous() && state->scalar_type() == at::kFloat &&
                    state->dim() == 3 && state->size(1) == taps - 1 && state->size(2) == C,
                "row_norm_add: fp32 state [slots, taps - 1, C]");
  }
  if (cw.has_value() || advance) {
    TORCH_CHECK(slot.has_value() && pos.has_value() && slot->scalar_type() == at::kInt &&
                    pos->scalar_type() == at::kInt && slot->numel() >= N && pos->numel() >= N &&
                    slot->is_contiguous() && pos->is_contiguous(),
                "row_norm_add: int32 slot / pos per row");
  }
  if (N == 0) return;
  const size_t lds = (size_t)(C + 5 * groups) * 4;
  TORCH_CHECK(lds <= 64 * 1024, "row_norm_add: row too wide");
  auto stream = at::hip::getCurrentHIPStream();
  pr_dispatch(dt, [&](auto* tag) {
    using T = std::remove_pointer_t<decltype(tag)>;
    auto ptr = [](c10::optional<torch::Tensor>& t) { return t.has_value() ? t->data_ptr() : nullptr; };
    auto run = [&](auto kernel, int threads, size_t bytes) {
      hipLaunchKernelGGL(kernel, dim3(N), dim3(threads), bytes, stream, (const int64_t*)ptr(tok), (const T*)ptr(table),
                         vocab, (const float*)ptr(x_in), (float*)ptr(x_out), (const T*)ptr(y), (const float*)ptr(pw),
                         (int)top, (const float*)ptr(nw), (int)groups, (float)eps, (const float*)ptr(cw), (int)taps,
                         (float*)ptr(state), (const int*)ptr(slot), (int*)ptr(pos), advance ? 1 : 0, (T*)ptr(h), (int)C);
    };
    bool vec = C <= 4096 && (C / groups) % 4 == 0;
    for (auto* o : {&table, &x_in, &x_out, &y, &nw, &cw, &state, &h})
      vec = vec && (!o->has_value() || reinterpret_cast<uintptr_t>((*o)->data_ptr()) % 16 == 0);
    const int wide = (int)((C / 4 + 63) / 64 * 64);
    auto conv = [&](auto kt) {
      constexpr int KT = decltype(kt)::value;
      cw.has_value() ? run(row_norm_add4_kernel<T, KT, true>, wide, 0) : run(row_norm_add4_kernel<T, KT, false>, wide, 0);
    };
    // a single expert's row is not read as four (1 x 4096: 3.5 us, so 3.1); rows of more than 512 threads: see the kernel's registers
    if (vec && !(y.has_value() && pw.has_value() && top > 0)) conv(std::integral_constant<int, 0>{});
    else if (vec && top == 1) conv(std::integral_constant<int, 1>{});
    else if (vec && (top <= 4 || (C > 2048 && cw.has_value()))) conv(std::integral_constant<int, 4>{});
    else if (vec) conv(std::integral_constant<int, 8>{});
    else run(row_norm_add_kernel<T>, kPrThreads, lds);
  });
}

void row_norm(torch::Tensor x, c10::optional<torch::Tensor> rows, torch::Tensor w, int64_t groups, double eps,
              torch::Tensor out) {
  PR_CHECK_DEV(x);
  PR_CHECK_DEV(out);
  PR_CHECK_DEV(w);
  const int64_t C = x.size(1), M = out.size(0);
  TORCH_CHECK(x.scalar_type() == at::kFloat && w.scalar_type() == at::kFloat && w.numel() == C && out.size(1) == C &&
                  groups >= 1 && C % groups == 0 && groups <= 1024,
              "row_norm: fp32 x [N, C], w [C]");
  if (rows.has_value()) {
    TORCH_CHECK(rows->is_cuda() && rows->scalar_type() == at::kInt && rows->numel() == M && rows->is_contiguous(),
                "row_norm: int32 rows");
  } else {
    TORCH_CHECK(M == x.size(0), "row_norm: one output row per input row");
  }
  if (M == 0) return;
  const size_t lds = (size_t)(C + 5 * groups) * 4;
  TORCH_CHECK(lds <= 64 * 1024, "row_norm: row too wide");
  pr_dispatch(out.scalar_type(), [&](auto* tag) {
    using T = std::remove_pointer_t<decltype(tag)>;
    hipLaunchKernelGGL(row_norm_kernel<T>, dim3(M), dim3(kPrThreads), lds, at::hip::getCurrentHIPStream(),
                       x.data_ptr<float>(), rows.has_value() ? rows->data_ptr<int>() : nullptr, w.data_ptr<float>(),
                       (int)groups, (float)eps, (T*)out.data_ptr(), (int)C);
  });
}

// h = x + conv(x) over packed rows, then the state of the step's sequences. The caller's descriptor
// (slot, pos, first per row; cu, seq_slot per sequence) comes from the state manager.
void conv_rows(torch::Tensor x, torch::Tensor cw, torch::Tensor state, torch::Tensor slot, torch::Tensor pos,
               torch::Tensor first, torch::Tensor cu, torch::Tensor seq_slot, torch::Tensor h) {
  PR_CHECK_DEV(x);
  PR_CHECK_DEV(cw);
  PR_CHECK_DEV(state);
  PR_CHECK_DEV(h);
  const int64_t N = x.size(0), C = x.size(1), taps = cw.size(0), S = seq_slot.numel();
  TORCH_CHECK(x.scalar_type() == at::kFloat && cw.scalar_type() == at::kFloat && state.scalar_type() == at::kFloat &&
                  cw.numel() == taps * C && h.numel() == N * C && taps <= kMaxTaps && state.dim() == 3 &&
                  state.size(1) == taps - 1 && state.size(2) == C,
              "conv_rows: shapes");
  for (auto* d : {&slot, &pos, &first, &cu, &seq_slot})
    TORCH_CHECK(d->is_cuda() && d->is_contiguous() && d->scalar_type() == at::kInt, "conv_rows: int32 descriptors");
  TORCH_CHECK(slot.numel() >= N && pos.numel() >= N && first.numel() >= N && cu.numel() == S + 1, "conv_rows: descriptors");
  if (N == 0) return;
  auto stream = at::hip::getCurrentHIPStream();
  pr_dispatch(h.scalar_type(), [&](auto* tag) {
    using T = std::remove_pointer_t<decltype(tag)>;
    auto run = [&](auto v) {
      constexpr int V = decltype(v)::value;
      const dim3 grid((N + 3) / 4, (C + 64 * V - 1) / (64 * V));
      hipLaunchKernelGGL((conv_rows_kernel<T, V>), grid, dim3(kPrThreads), 0, stream, x.data_ptr<float>(),
                         cw.data_ptr<float>(), (int)taps, state.data_ptr<float>(), slot.data_ptr<int>(),
                         pos.data_ptr<int>(), first.data_ptr<int>(), (T*)h.data_ptr(), (int)N, (int)C);
    };
    if (C % 4 == 0) run(std::integral_constant<int, 4>{});
    else  // any width
      run(std::integral_constant<int, 1>{});
  });
  if (taps > 1)
    hipLaunchKernelGGL(conv_state_kernel, dim3(S, (C + kPrThreads - 1) / kPrThreads), dim3(kPrThreads), 0, stream,
                       x.data_ptr<float>(), (int)taps, state.data_ptr<float>(), cu.data_ptr<int>(),
                       seq_slot.data_ptr<int>(), (int)C);
}

// x_out = x + norm(y) and h = x_out + conv(x_out) over packed rows, then the state, as
// row_norm_add and conv_rows do one after the other; x and x_out differ. Groups of 256 or 512 channels and at most
// 4 taps (norm_conv_kernel).
void norm_conv_rows(torch::Tensor x, torch::Tensor x_out, torch::Tensor y, torch::Tensor nw, int64_t groups,
                    double eps, torch::Tensor cw, torch::Tensor state, torch::Tensor slot, torch::Tensor pos,
                    torch::Tensor first, torch::Tensor cu, torch::Tensor seq_slot, torch::Tensor h) {
  for (auto* o : {&x, &x_out, &y, &nw, &cw, &state, &h}) {
    PR_CHECK_DEV(*o);
    TORCH_CHECK(reinterpret_cast<uintptr_t>(o->data_ptr()) % 16 == 0, "norm_conv_rows: 16-byte alignment");
  }
  const int64_t N = x.size(0), C = x.size(1), taps = cw.size(0), S = seq_slot.numel();
  for (auto* o : {&x, &x_out, &nw, &cw, &state})
    TORCH_CHECK(o->scalar_type() == at::kFloat, "norm_conv_rows: fp32 x, weights, taps and state");
  TORCH_CHECK(x_out.numel() == N * C && h.numel() == N * C && nw.numel() == C && cw.numel() == taps * C &&
                  y.scalar_type() == h.scalar_type() && state.dim() == 3 && state.size(1) == taps - 1 &&
                  state.size(2) == C,
              "norm_conv_rows: shapes");
  TORCH_CHECK(N == 0 || x.data_ptr() != x_out.data_ptr(), "norm_conv_rows: x_out is another buffer than x");
  const int64_t quarters = groups > 0 && C % (256 * groups) == 0 ? C / (256 * groups) : 0;
  TORCH_CHECK((quarters == 1 || quarters == 2) && taps >= 1 && taps <= kNcTaps,
              "norm_conv_rows: groups of 256 or 512 channels, up to 4 taps");
  TORCH_CHECK(y.numel() == N * C, "norm_conv_rows: y rows");
  for (auto* d : {&slot, &pos, &first, &cu, &seq_slot})
    TORCH_CHECK(d->is_cuda() && d->is_contiguous() && d->scalar_type() == at::kInt, "norm_conv_rows: int32 descriptors");
  TORCH_CHECK(slot.numel() >= N && pos.numel() >= N && first.numel() >= N && cu.numel() == S + 1,
              "norm_conv_rows: descriptors");
  if (N == 0) return;
  auto stream = at::hip::getCurrentHIPStream();
  pr_dispatch(h.scalar_type(), [&](auto* tag) {
    using T = std::remove_pointer_t<decltype(tag)>;
    auto run = [&](auto quarter) {
      constexpr int Q = decltype(quarter)::value;
      // 4·n - 3 rows a wave, so that they and the three before them are whole fours: 5 while the chip (256 CUs) holds
      // all workgroups at once, then as many as keep it so up to 37, then as many in whole rounds. 8192 rows of 2048
      // in 4 groups, one round of 512 workgroups from 17: 5 48 us, 13 44, 21 38, 29 44, 61 56; 1024 rows: 11, 17, 21.
      const int64_t gy = (groups + 3) / 4, slots = 256 * norm_conv_blocks<Q>();
      const int64_t rounds = (N * gy + 37 * slots - 1) / (37 * slots);
      const int64_t rows = (N * gy + rounds * slots - 1) / (rounds * slots);
      const int span = (int)std::max<int64_t>(5, (rows + 6) / 4 * 4 - 3);
      hipLaunchKernelGGL((norm_conv_kernel<T, Q>), dim3((N + span - 1) / span, gy), dim3(kPrThreads), 0, stream,
                         x.data_ptr<float>(), x_out.data_ptr<float>(), (const T*)y.data_ptr(), nw.data_ptr<float>(),
                         (int)groups, (float)eps, cw.data_ptr<float>(), (int)taps, state.data_ptr<float>(),
                         slot.data_ptr<int>(), pos.data_ptr<int>(), first.data_ptr<int>(), (T*)h.data_ptr(), (int)N,
                         (int)C, span);
    };
    if (quarters == 1) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 2>{});
  });
  if (taps > 1)
    hipLaunchKernelGGL(conv_state_kernel, dim3(S, (C + kPrThreads - 1) / kPrThreads), dim3(kPrThreads), 0, stream,
                       x_out.data_ptr<float>(), (int)taps, state.data_ptr<float>(), cu.data_ptr<int>(),
                       seq_slot.data_ptr<int>(), (int)C);
}

// x (fp32 [N, C]) from token ids and tables, or x_in + the sublayer's output; h = rms_norm(x)·nw.
// ya [N, C] (or [N·top, C] with pw [N, top (+ 1 with ys)]), yb [N, C]; wa / wb fp32 norm weights. advance:
// pos (int32 [N]) is incremented first; the position rows are taken at pos.
void residual_norm(c10::optional<torch::Tensor> tok, c10::optional<torch::Tensor> table,
                   c10::optional<torch::Tensor> ptable, c10::optional<torch::Tensor> x_in,
                   c10::optional<torch::Tensor> x_out, c10::optional<torch::Tensor> ya, c10::optional<torch::Tensor> wa,
                   c10::optional<torch::Tensor> yb, c10::optional<torch::Tensor> wb, double coef, double yeps,
                   c10::optional<torch::Tensor> pw, c10::optional<torch::Tensor> ys, c10::optional<torch::Tensor> nw,
                   double eps, c10::optional<torch::Tensor> pos, bool advance, c10::optional<torch::Tensor> h) {
  TORCH_CHECK(tok.has_value() != x_in.has_value(), "residual_norm: token ids or x_in");
  TORCH_CHECK(x_out.has_value() || h.has_value(), "residual_norm: nothing to write");
  TORCH_CHECK(h.has_value() == nw.has_value(), "residual_norm: h and its norm weight");
  TORCH_CHECK(!yb.has_value() || (ya.has_value() && !pw.has_value()), "residual_norm: yb beside ya");
  TORCH_CHECK(!ys.has_value() || pw.has_value(), "residual_norm: a shared row goes with expert rows");
  for (auto* o : {&tok, &table, &ptable, &x_in, &x_out, &ya, &wa, &yb, &wb, &pw, &ys, &nw, &h})
    if (o->has_value()) PR_CHECK_DEV(**o);
  at::ScalarType dt = at::kFloat;
  int64_t N, C, vocab = 0, npos = 0;
  if (tok.has_value()) {
    TORCH_CHECK(table.has_value() && tok->scalar_type() == at::kLong && table->dim() == 2,
                "residual_norm: int64 ids and their table");
    N = tok->numel();
    C = table->size(1);
    vocab = table->size(0);
    dt = table->scalar_type();
    if (ptable.has_value()) {
      npos = ptable->size(0);
      TORCH_CHECK(ptable->dim() == 2 && ptable->size(1) == C && ptable->scalar_type() == dt && npos > 0,
                  "residual_norm: position table [positions, C]");
    }
  } else {
    TORCH_CHECK(x_in->dim() == 2, "residual_norm: x_in [N, C]");
    N = x_in->size(0);
    C = x_in->size(1);
    if (ya.has_value()) dt = ya->scalar_type();
    else if (h.has_value()) dt = h->scalar_type();
  }
  for (auto* o : {&x_in, &x_out})
    TORCH_CHECK(!o->has_value() || ((*o)->scalar_type() == at::kFloat && (*o)->numel() == N * C),
                "residual_norm: x is fp32 [N, C]");
  for (auto* o : {&wa, &wb, &nw})
    TORCH_CHECK(!o->has_value() || ((*o)->scalar_type() == at::kFloat && (*o)->numel() == C),
                "residual_norm: fp32 weights [C]");
  for (auto* o : {&yb, &ys, &h})
    TORCH_CHECK(!o->has_value() || ((*o)->scalar_type() == dt && (*o)->numel() == N * C), "residual_norm: rows [N, C]");
  int64_t top = 1, pws = 1;
  if (pw.has_value()) {
    pws = pw->size(1);
    top = pws - (ys.has_value() ? 1 : 0);
    TORCH_CHECK(pw->dim() == 2 && pw->size(0) == N && pw->scalar_type() == at::kFloat && top >= 1 && !wa.has_value(),
                "residual_norm: fp32 weights per expert row");
  }
  TORCH_CHECK(!ya.has_value() || (ya->scalar_type() == dt && ya->numel() == N * top * C), "residual_norm: ya rows");
  if (advance || ptable.has_value())
    TORCH_CHECK(pos.has_value() && pos->is_cuda() && pos->is_contiguous() && pos->scalar_type() == at::kInt &&
                    pos->numel() >= N,
                "residual_norm: int32 position per row");
  if (N == 0) return;
  bool vec = C % 4 == 0;
  for (auto* o : {&table, &ptable, &x_in, &x_out, &ya, &wa, &yb, &wb, &ys, &nw, &h})
    vec = vec && (!o->has_value() || reinterpret_cast<uintptr_t>((*o)->data_ptr()) % 16 == 0);
  const int64_t groups = vec ? C / 4 : C;  // vectors per row
  TORCH_CHECK(groups <= 4096, "residual_norm: row too wide");
  const int threads = (int)std::min<int64_t>(1024, (groups + 63) / 64 * 64);
  pr_dispatch(dt, [&](auto* tag) {
    using T = std::remove_pointer_t<decltype(tag)>;
    auto ptr = [](c10::optional<torch::Tensor>& t) { return t.has_value() ? t->data_ptr() : nullptr; };
    ResidualArgs<T> a{(const int64_t*)ptr(tok), (const T*)ptr(table), (const T*)ptr(ptable), vocab, npos,
                      (const float*)ptr(x_in), (float*)ptr(x_out), (const T*)ptr(ya), (const T*)ptr(yb),
                      (const float*)ptr(wa), (const float*)ptr(wb), (float)coef, (float)yeps, (const float*)ptr(pw),
                      (int)top, (int)pws, (const T*)ptr(ys), (const float*)ptr(nw), (float)eps, (int*)ptr(pos),
                      advance ? 1 : 0, (T*)ptr(h), (int)C};
    auto run = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(N), dim3(threads), 0, at::hip::getCurrentHIPStream(), a); };
    if (vec && groups > 1024) run(residual_norm_kernel<T, 4, 4, 4>);
    else if (vec && sizeof(T) == 4 && groups > 512) run(residual_norm_kernel<T, 4, 1, 4>);
    else if (vec) run(residual_norm_kernel<T, 4, 1, 8>);
    else if (groups <= 1024) run(residual_norm_kernel<T, 1, 1, 8>);
    else run(residual_norm_kernel<T, 1, 4, 4>);
  });
}
