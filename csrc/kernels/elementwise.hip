// Memory-bound kernels: GELU fwd/bwd (+ fused bias-gradient column sum), gated-MLP
// activation, column sums, token+position embedding fwd/bwd, RoPE on fused QKV, int8 KV
// quantisation, and on-device tensor statistics (moments, min/max, density histogram).
//
// All streams use 16-B per-lane vectors (8 bf16 or 4 fp32), grid-stride loops capped at
// 8192 workgroups for the large passes (2048 elsewhere; CDNA HIP guide, Guideline 11/13). Column-sum fusions keep each thread's
// 8 columns fixed while it walks rows, so the partial sums live in registers; a workgroup
// reduces its 4 waves in LDS and writes one partial row, finished by a tiny reduction.
#include "common.h"
#include "deferred.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <cstdlib>

namespace penroz {

__device__ __forceinline__ float act_grad_f(float x, int kind) {
  if (kind == 2) {
    const float s = 1.f / (1.f + __expf(-x));
    return s * (1.f + x * (1.f - s));
  }
  return gelu_grad_f(x, kind);
}

template <typename T, bool NT = false>
__global__ void __launch_bounds__(256) gelu_fwd_kernel(const T* __restrict__ x, T* __restrict__ y, int64_t n8,
                                                       int approx) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n8; i += (int64_t)gridDim.x * blockDim.x) {
    float v[8];
    load8<NT>(x + 8 * i, v);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = gelu_f(v[k], approx);
    store8<NT>(y + 8 * i, v);
  }
}

template <typename T, bool NT = false>
__global__ void __launch_bounds__(256) gelu_bwd_kernel(const T* __restrict__ dy, const T* __restrict__ x,
                                                       T* __restrict__ dx, int64_t n8, int approx) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n8; i += (int64_t)gridDim.x * blockDim.x) {
    float g[8], v[8];
    load8<NT>(dy + 8 * i, g);
    load8<NT>(x + 8 * i, v);
#pragma unroll
    for (int k = 0; k < 8; ++k) g[k] *= gelu_grad_f(v[k], approx);
    store8<NT>(dx + 8 * i, g);
  }
}

// MODE 0: colsum of x.  MODE 1: dx = dy*gelu'(x) written to out, colsum of dx.
// grid = (F/512 column tiles, R row splits); block 256 = 4 waves; lane -> 8 columns.
template <int MODE, typename T, bool NT = false>
__global__ void __launch_bounds__(256) rows_colsum_kernel(const T* __restrict__ a, const T* __restrict__ x,
                                                          T* __restrict__ out, float* __restrict__ part, int N, int F,
                                                          int approx) {
  __shared__ float red[4][512];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int col = blockIdx.x * 512 + 8 * lane;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const bool active = col < F;
  const int R = gridDim.y;
  const int rows_per = (N + R - 1) / R;
  const int r0 = blockIdx.y * rows_per, r1 = min(N, r0 + rows_per);
  if (active) {
    for (int r = r0 + wid; r < r1; r += 4) {
      const size_t off = (size_t)r * F + col;
      float v[8];
      load8<NT>(a + off, v);
      if constexpr (MODE == 1) {
        float xv[8];
        load8<NT>(x + off, xv);
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = to_f(from_f<T>(v[k] * gelu_grad_f(xv[k], approx)));
        // v now holds the *rounded* values: dbias matches the bf16 gradient the GEMMs see
        store8<NT>(out + off, v);
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) acc[k] += v[k];
    }
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) red[wid][8 * lane + k] = acc[k];
  __syncthreads();
  for (int c = threadIdx.x; c < 512; c += 256) {
    const int gc = blockIdx.x * 512 + c;
    if (gc < F) part[(size_t)blockIdx.y * F + gc] = red[0][c] + red[1][c] + red[2][c] + red[3][c];
  }
}

// ------------------------------------------------------------------------------ gated MLP act
template <typename T, bool NT = false>
__global__ void __launch_bounds__(256) gated_fwd_kernel(const T* __restrict__ g, const T* __restrict__ u,
                                                        T* __restrict__ y, int64_t n8, int kind) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n8; i += (int64_t)gridDim.x * blockDim.x) {
    float gv[8], uv[8];
    load8<NT>(g + 8 * i, gv);
    load8<NT>(u + 8 * i, uv);
#pragma unroll
    for (int k = 0; k < 8; ++k) gv[k] = act_f(gv[k], kind) * uv[k];
    store8<NT>(y + 8 * i, gv);
  }
}

// decode: gate and up halves of one fused [N, 2I] projection -> act(gate) * up [N, I]
template <typename T, bool NT = false>
__global__ void __launch_bounds__(256) gated_packed_kernel(const T* __restrict__ gu, T* __restrict__ y, int64_t n8,
                                                           int I8, int kind) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n8; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / I8, c = i - r * I8;
    float gv[8], uv[8];
    load8<NT>(gu + 8 * (r * 2 * I8 + c), gv);
    load8<NT>(gu + 8 * (r * 2 * I8 + I8 + c), uv);
#pragma unroll
    for (int k = 0; k < 8; ++k) gv[k] = act_f(gv[k], kind) * uv[k];
    store8<NT>(y + 8 * i, gv);
  }
}

template <typename T, bool NT = false>
__global__ void __launch_bounds__(256) gated_bwd_kernel(const T* __restrict__ dy, const T* __restrict__ g,
                                                        const T* __restrict__ u, T* __restrict__ dg,
                                                        T* __restrict__ du, int64_t n8, int kind) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n8; i += (int64_t)gridDim.x * blockDim.x) {
    float d[8], gv[8], uv[8], o1[8], o2[8];
    load8<NT>(dy + 8 * i, d);
    load8<NT>(g + 8 * i, gv);
    load8<NT>(u + 8 * i, uv);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      o1[k] = d[k] * uv[k] * act_grad_f(gv[k], kind);
      o2[k] = d[k] * act_f(gv[k], kind);
    }
    store8<NT>(dg + 8 * i, o1);
    store8<NT>(du + 8 * i, o2);
  }
}

// packed form of the backward: gu = [gate | up] per row (I8 chunks of 8 each), dgu likewise —
// the layout one GEMM over the concatenated [gate; up] weight consumes (fused Gemma executor)
template <typename T, bool NT = false>
__global__ void __launch_bounds__(256) gated_bwd_packed_kernel(const T* __restrict__ dy, const T* __restrict__ gu,
                                                               T* __restrict__ dgu, int64_t n8, int I8, int kind) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n8; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / I8, c = i - r * I8;
    const int64_t go = 8 * (r * 2 * I8 + c), uo = go + 8 * (int64_t)I8;
    float d[8], gv[8], uv[8], o1[8], o2[8];
    load8<NT>(dy + 8 * i, d);
    load8<NT>(gu + go, gv);
    load8<NT>(gu + uo, uv);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      o1[k] = d[k] * uv[k] * act_grad_f(gv[k], kind);
      o2[k] = d[k] * act_f(gv[k], kind);
    }
    store8<NT>(dgu + go, o1);
    store8<NT>(dgu + uo, o2);
  }
}

// ------------------------------------------------------------------------------ embedding
// out[n, :] = wte[idx[n], :] + wpe[off + n % T, :]   (one wave per token row, 16-B lanes)
template <typename TW>
__global__ void __launch_bounds__(256) embed_fwd_kernel(const int64_t* __restrict__ idx, const TW* __restrict__ wte,
                                                        const TW* __restrict__ wpe, float* __restrict__ out, int N,
                                                        int T, int C, int off, int V, const int64_t* __restrict__ off_dev,
                                                        int P, uint64_t dseed, float dp) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= N) return;
  int64_t tok = idx[row];
  PZ_DEVICE_CHECK(tok >= 0 && tok < V);
  tok = tok < 0 ? 0 : (tok >= V ? V - 1 : tok);
  if (off_dev != nullptr) off = (int)*off_dev;  // graph-replayed decode: position on the device
  const int pos = min(off + row % T, P - 1);
  for (int c = 8 * lane; c < C; c += 512) {
    float a[8], b[8];
    Vec8<TW>::load(wte + (size_t)tok * C + c, a);
    Vec8<TW>::load(wpe + (size_t)pos * C + c, b);
#pragma unroll
    for (int k = 0; k < 8; ++k) a[k] += b[k];
    if (dp > 0.f) {  // embedding dropout (HF GPT-2 embd_pdrop); the backward regenerates the mask
      const float inv = 1.f / (1.f - dp);
#pragma unroll
      for (int k = 0; k < 8; ++k) a[k] *= dropout_mult(dseed, (size_t)row * C + c + k, dp, inv);
    }
    Vec8<float>::store(out + (size_t)row * C + c, a);
  }
}

// out [C][R] = in [R][C]ᵀ, bf16, 64×64 tiles through LDS (16-B global loads and stores). Used
// for the weight copies of the data-gradient GEMMs (dx = dy·W runs ~12-22 % faster on
// hipBLASLt with W stored transposed: both operands then reduction-contiguous, the forward's
// layout — profiles/dgrad_layout_r1.log).
struct Transpose {
  const uint16_t* in;
  uint16_t* out;
  int R, C, tile0;  // tile0: tiles of the matrices before
};
constexpr int kTransposes = 64;
struct Transposes {
  Transpose m[kTransposes];
  int n;
};

// All copies of a step in one launch: by themselves GPT-2's 49 take 3 to 4 us each, little above an empty launch, and 5 us of the
// host's time. A workgroup finds its matrix by halving.
__global__ void __launch_bounds__(256) transpose_bf16_kernel(const Transposes all) {
  __shared__ uint16_t tile[64][66];
  int lo = 0, hi = all.n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((int)blockIdx.x >= all.m[mid].tile0) lo = mid;
    else hi = mid - 1;
  }
  const uint16_t* __restrict__ in = all.m[lo].in;
  uint16_t* __restrict__ out = all.m[lo].out;
  const int R = all.m[lo].R, C = all.m[lo].C, id = blockIdx.x - all.m[lo].tile0;
  const int tiles_c = C / 64;
  const int r0 = (id / tiles_c) * 64, c0 = (id % tiles_c) * 64;
  const int t = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int v = t + 256 * i, row = v >> 3, ch = v & 7;
    const uint4 u = *reinterpret_cast<const uint4*>(in + (size_t)(r0 + row) * C + c0 + 8 * ch);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      tile[row][8 * ch + 2 * j] = (uint16_t)(w[j] & 0xffff);
      tile[row][8 * ch + 2 * j + 1] = (uint16_t)(w[j] >> 16);
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int v = t + 256 * i, orow = v >> 3, ch = v & 7;  // output row = input column c0 + orow
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      w[j] = (uint32_t)tile[8 * ch + 2 * j][orow] | ((uint32_t)tile[8 * ch + 2 * j + 1][orow] << 16);
    *reinterpret_cast<uint4*>(out + (size_t)(c0 + orow) * R + r0 + 8 * ch) = uint4{w[0], w[1], w[2], w[3]};
  }
}

// dwte[idx[n]] += dout[n]  (fp32 atomics; each wave instruction = 256 contiguous bytes)
__global__ void __launch_bounds__(256) embed_bwd_tok_kernel(const float* __restrict__ dout,
                                                            const int64_t* __restrict__ idx,
                                                            float* __restrict__ dwte, int N, int C, int V,
                                                            uint64_t dseed, float dp) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= N) return;
  const int64_t tok = idx[row];
  PZ_DEVICE_CHECK(tok >= 0 && tok < V);
  if (tok < 0 || tok >= V) return;
  float* dst = dwte + (size_t)tok * C;
  const float* src = dout + (size_t)row * C;
  if (dp > 0.f) {
    const float inv = 1.f / (1.f - dp);
    for (int c = lane; c < C; c += 64)
      atomicAdd(dst + c, src[c] * dropout_mult(dseed, (size_t)row * C + c, dp, inv));
  } else {
    for (int c = lane; c < C; c += 64) atomicAdd(dst + c, src[c]);
  }
}

// dwpe[off + t] += Σ_b dout[b*T + t]   (one workgroup per position, no atomics)
__global__ void __launch_bounds__(256) embed_bwd_pos_kernel(const float* __restrict__ dout, float* __restrict__ dwpe,
                                                            int B, int T, int C, int off, uint64_t dseed, float dp) {
  const int t = blockIdx.x;
  const float inv = dp > 0.f ? 1.f / (1.f - dp) : 1.f;
  for (int c = threadIdx.x * 4; c < C; c += 1024) {
    float4_t s = {0.f, 0.f, 0.f, 0.f};
    for (int b = 0; b < B; ++b) {
      const size_t e = ((size_t)b * T + t) * C + c;
      float4_t g = *reinterpret_cast<const float4_t*>(dout + e);
      if (dp > 0.f) {
#pragma unroll
        for (int k = 0; k < 4; ++k) g[k] *= dropout_mult(dseed, e + k, dp, inv);
      }
      s += g;
    }
    float4_t* d = reinterpret_cast<float4_t*>(dwpe + (size_t)(off + t) * C + c);
    *d = *d + s;
  }
}

// ------------------------------------------------------------------------------ RoPE
// qkv [B*T, (H+2Hkv)*D]; rotate the first H+Hkv heads (Q and K); V copied. cos/sin [T, D/2].
template <typename T>
__global__ void __launch_bounds__(256) rope_kernel(const T* __restrict__ in, T* __restrict__ out,
                                                   const float* __restrict__ cosv, const float* __restrict__ sinv,
                                                   int64_t rows, int Tlen, int H, int Hkv, int D, int inverse) {
  const int W = (H + 2 * Hkv) * D;
  const int half = D / 2;
  const int64_t total = rows * (int64_t)W;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / W;
    const int c = (int)(i - r * W);
    const int head = c / D;
    const int d = c - head * D;
    if (head >= H + Hkv) {
      out[i] = in[i];
      continue;
    }
    const int t = (int)(r % Tlen);
    const int j = d < half ? d : d - half;
    const float cs = cosv[(size_t)t * half + j];
    float sn = sinv[(size_t)t * half + j];
    if (inverse) sn = -sn;
    const int64_t hb = r * W + (int64_t)head * D;
    const float x1 = to_f(in[hb + j]), x2 = to_f(in[hb + j + half]);
    const float o = d < half ? (x1 * cs - x2 * sn) : (x2 * cs + x1 * sn);
    out[i] = from_f<T>(o);
  }
}

// cos / sin [T, n] of positions *pos + i, one launch instead of a dozen elementwise ones per decode step (4.5 us each in a
// replayed step: 30 us a token of Gemma-3 1B), in their arithmetic
__global__ void __launch_bounds__(256) rope_table_kernel(const float* __restrict__ inv, const int64_t* __restrict__ pos,
                                                         float* __restrict__ cosv, float* __restrict__ sinv, int T, int n) {
  const float p = (float)*pos;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < T * n; i += gridDim.x * 256) {
    const int t = i / n;
    const float a = (p + (float)t) * inv[i - t * n];
    cosv[i] = cosf(a);
    sinv[i] = sinf(a);
  }
}

// Vectorised form (D % 16 == 0, contiguous fp32 cos / sin tables): one work item = 8 rotated pairs
// (16-B loads of both halves and of cos / sin) or one 16-B chunk of the V columns copied through;
// the scalar kernel above did a 64-bit division, two gathered 2-B loads and a 2-B store per element
// (≈ 0.6 TB/s at Gemma-3 1B shapes).
template <typename T>
__global__ void __launch_bounds__(256) rope_vec_kernel(const T* __restrict__ in, T* __restrict__ out,
                                                       const float* __restrict__ cosv,
                                                       const float* __restrict__ sinv, int64_t rows, int Tlen,
                                                       int H, int Hkv, int D, int inverse) {
  const int W = (H + 2 * Hkv) * D, half = D / 2, h8 = half / 8;
  const int nrot = (H + Hkv) * h8, per = nrot + Hkv * D / 8;
  const int64_t total = rows * (int64_t)per;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / per;
    const int k = (int)(i - r * per);
    if (k < nrot) {
      const int head = k / h8, j0 = 8 * (k - head * h8);
      const int t = (int)(r % Tlen);
      const int64_t base = r * W + (int64_t)head * D;
      float x1[8], x2[8];
      Vec8<T>::load(in + base + j0, x1);
      Vec8<T>::load(in + base + half + j0, x2);
      const float* cp = cosv + (size_t)t * half + j0;
      const float* sp = sinv + (size_t)t * half + j0;
      const float4 c0 = *reinterpret_cast<const float4*>(cp), c1 = *reinterpret_cast<const float4*>(cp + 4);
      const float4 s0 = *reinterpret_cast<const float4*>(sp), s1 = *reinterpret_cast<const float4*>(sp + 4);
      const float cs[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
      float sn[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
      float o1[8], o2[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (inverse) sn[e] = -sn[e];
        o1[e] = x1[e] * cs[e] - x2[e] * sn[e];
        o2[e] = x2[e] * cs[e] + x1[e] * sn[e];
      }
      Vec8<T>::store(out + base + j0, o1);
      Vec8<T>::store(out + base + half + j0, o2);
    } else {
      const int64_t off = r * W + (int64_t)(H + Hkv) * D + 8 * (k - nrot);
      float v[8];
      Vec8<T>::load(in + off, v);
      Vec8<T>::store(out + off, v);
    }
  }
}

// A prompt's new keys and values from qkv [B, T, (H + 2 Hkv) * D] into the caches [B, Hkv, cap, D] at pos.., and with ROPE the
// rotated queries into q [B, T, H, D] (keys rotated on the way, angles in the arithmetic of rope_table_kernel). Bound by the
// host: a layer's pass was the table (7 launches of 5 us of host time each), the rotation, two strided copies. A workgroup takes
// `per_wg` tokens, whose angles it computes once for all heads into LDS; an item is 8 rotated pairs or 16 bytes copied. 3 x 200
// tokens, 4 + 1 heads of 256: 5.1 us of the device for the former 25.
template <bool ROPE, typename F>
__global__ void __launch_bounds__(256) prompt_kv_kernel(const __hip_bfloat16* __restrict__ in, const F* __restrict__ inv,
                                                        __hip_bfloat16* __restrict__ q, __hip_bfloat16* __restrict__ kc,
                                                        __hip_bfloat16* __restrict__ vc, int64_t tokens, int per_wg, int T,
                                                        int H, int Hkv, int D, int64_t cap, int pos) {
  extern __shared__ float angles[];  // [per_wg][cos D/2, sin D/2]
  const int half = D / 2, h8 = half / 8, d8 = D / 8;
  const int64_t row0 = blockIdx.x * (int64_t)per_wg, W = (int64_t)(H + 2 * Hkv) * D;
  const int n = (int)(tokens - row0 < per_wg ? tokens - row0 : per_wg);
  if (ROPE) {
    for (int i = threadIdx.x; i < n * half; i += 256) {
      const int r = i / half, j = i - r * half;
      const float a = (float)(pos + (int)((row0 + r) % T)) * to_f(inv[j]);
      angles[r * D + j] = cosf(a);
      angles[r * D + half + j] = sinf(a);
    }
    __syncthreads();
  }
  const int nrot = ROPE ? (H + Hkv) * h8 : 0, ncopy = (ROPE ? Hkv : 2 * Hkv) * d8, per = nrot + ncopy;
  for (int i = threadIdx.x; i < n * per; i += 256) {
    const int r = i / per, k = i - r * per;
    const int64_t row = row0 + r, b = row / T, slot = pos + row - b * T;
    const __hip_bfloat16* src = in + row * W;
    if (ROPE && k < nrot) {
      const int head = k / h8, j0 = 8 * (k - head * h8);
      const float *cs = angles + r * D + j0, *sn = cs + half;
      float x1[8], x2[8], o1[8], o2[8];
      Vec8<__hip_bfloat16>::load(src + (int64_t)head * D + j0, x1);
      Vec8<__hip_bfloat16>::load(src + (int64_t)head * D + half + j0, x2);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        o1[e] = x1[e] * cs[e] - x2[e] * sn[e];
        o2[e] = x2[e] * cs[e] + x1[e] * sn[e];
      }
      __hip_bfloat16* dst = head < H ? q + (row * H + head) * D : kc + ((b * Hkv + head - H) * cap + slot) * D;
      Vec8<__hip_bfloat16>::store(dst + j0, o1);
      Vec8<__hip_bfloat16>::store(dst + half + j0, o2);
    } else {
      const int c = k - nrot, head = c / d8, j0 = 8 * (c - head * d8), kv = ROPE ? head + Hkv : head;  // kv: of the k heads, then v
      const uint4 x = *reinterpret_cast<const uint4*>(src + (int64_t)(H + kv) * D + j0);
      __hip_bfloat16* dst = (kv < Hkv ? kc : vc) + ((b * Hkv + (kv < Hkv ? kv : kv - Hkv)) * cap + slot) * D;
      *reinterpret_cast<uint4*>(dst + j0) = x;
    }
  }
}

// ------------------------------------------------------------------------------ int8 KV quant
// x [B, T, Hkv, D] -> q [B, Hkv, cap, D] int8 at pos.., scale [B, Hkv, cap] f32 (absmax/127)
template <typename T>
__global__ void __launch_bounds__(256) kv_quant_kernel(const T* __restrict__ x, int8_t* __restrict__ q,
                                                       float* __restrict__ scale, int Bn, int Tn, int Hkv, int D,
                                                       int cap, int pos) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);  // over B*T*Hkv
  if (row >= Bn * Tn * Hkv) return;
  const int h = row % Hkv;
  const int t = (row / Hkv) % Tn;
  const int b = row / (Hkv * Tn);
  const T* src = x + (size_t)row * D;
  float m = 0.f;
  for (int d = lane; d < D; d += 64) m = fmaxf(m, fabsf(to_f(src[d])));
  m = wave_max(m);
  float s = m / 127.f;
  if (s == 0.f) s = 1.f;
  const size_t slot = ((size_t)b * Hkv + h) * cap + pos + t;
  for (int d = lane; d < D; d += 64) {
    float v = rintf(to_f(src[d]) / s);
    v = fminf(fmaxf(v, -128.f), 127.f);
    q[slot * D + d] = (int8_t)v;
  }
  if (lane == 0) scale[slot] = s;
}

// ------------------------------------------------------------------------------ stats
// pass 1: per-block (sum, min, max); pass 2: per-block Σ(x-mean)^2 + LDS histogram.
template <typename T>
__global__ void __launch_bounds__(256) stats_pass1_kernel(const T* __restrict__ x, int64_t n,
                                                          float* __restrict__ part) {
  __shared__ float red[3][4];
  float s = 0.f, mn = INFINITY, mx = -INFINITY;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float v = to_f(x[i]);
    s += v;
    mn = fminf(mn, v);
    mx = fmaxf(mx, v);
  }
  s = wave_sum(s);
  mn = wave_min(mn);
  mx = wave_max(mx);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { red[0][w] = s; red[1][w] = mn; red[2][w] = mx; }
  __syncthreads();
  if (threadIdx.x == 0) {
    part[blockIdx.x * 3 + 0] = red[0][0] + red[0][1] + red[0][2] + red[0][3];
    part[blockIdx.x * 3 + 1] = fminf(fminf(red[1][0], red[1][1]), fminf(red[1][2], red[1][3]));
    part[blockIdx.x * 3 + 2] = fmaxf(fmaxf(red[2][0], red[2][1]), fmaxf(red[2][2], red[2][3]));
  }
}

template <typename T>
__global__ void __launch_bounds__(256) stats_pass2_kernel(const T* __restrict__ x, int64_t n,
                                                          const float* __restrict__ mmm,  // mean, lo, hi
                                                          float* __restrict__ part, float* __restrict__ hist,
                                                          int bins) {
  extern __shared__ __attribute__((aligned(16))) float lh[];
  __shared__ float red[4];
  for (int b = threadIdx.x; b < bins; b += blockDim.x) lh[b] = 0.f;
  __syncthreads();
  const float mean = mmm[0], lo = mmm[1], hi = mmm[2];
  const float inv = bins / (hi - lo);
  float ss = 0.f;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float v = to_f(x[i]);
    ss += (v - mean) * (v - mean);
    int b = (int)((v - lo) * inv);
    b = b < 0 ? 0 : (b >= bins ? bins - 1 : b);
    atomicAdd(&lh[b], 1.f);
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
  for (int b = threadIdx.x; b < bins; b += blockDim.x)
    if (lh[b] != 0.f) atomicAdd(&hist[b], lh[b]);
}

}  // namespace penroz

// ============================================================================ host side
using namespace penroz;

#define FOR_FLOAT_TYPES(t, NAME, ...)                                               \
  if ((t) == torch::kFloat32) { using NAME = float; __VA_ARGS__; }                  \
  else if ((t) == torch::kBFloat16) { using NAME = bf16; __VA_ARGS__; }             \
  else if ((t) == torch::kFloat16) { using NAME = __half; __VA_ARGS__; }            \
  else TORCH_CHECK(false, "unsupported dtype");

// PENROZ_EW_NT (non-temporal loads / stores, default on) and PENROZ_EW_GRID (workgroup cap of the
// grid-stride launches, default 8192) for the large streaming passes: GELU, gated activation,
// GELU backward + bias columns. Against the old plain / 2048 setting (profiles/ew_ab_r4.log):
// gelu_fwd 180-198 -> 146-152 us, GELU backward + columns 292 -> 246 us (GPT-2 shapes), gated
// forward 68 -> 58 us, gated backward 129 -> 109 us (Gemma-3 1B shapes).
static bool ew_nt() {
  const char* e = std::getenv("PENROZ_EW_NT");
  return e && *e ? std::atoi(e) != 0 : true;
}
static int ew_cap() {
  const char* e = std::getenv("PENROZ_EW_GRID");
  return e && *e ? std::max(1, std::atoi(e)) : 8192;
}

static inline int grid_for(int64_t work, int block = 256, int cap = 2048) {
  int64_t g = (work + block - 1) / block;
  return (int)std::max<int64_t>(1, std::min<int64_t>(g, cap));
}

static void check_vec8(const torch::Tensor& t) {
  TORCH_CHECK(t.is_cuda() && t.is_contiguous(), "expected a contiguous GPU tensor");
  TORCH_CHECK(t.numel() % 8 == 0, "element count must be a multiple of 8");
  TORCH_CHECK(reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0, "tensor must be 16-byte aligned");
}

void gelu_fwd(torch::Tensor x, int64_t approx, torch::Tensor y) {
  check_vec8(x);
  check_vec8(y);
  TORCH_CHECK(x.scalar_type() == y.scalar_type() && x.numel() == y.numel());
  const int64_t n8 = x.numel() / 8;
  auto stream = at::hip::getCurrentHIPStream();
  FOR_FLOAT_TYPES(x.scalar_type(), T,
    hipLaunchKernelGGL((ew_nt() ? gelu_fwd_kernel<T, true> : gelu_fwd_kernel<T, false>), dim3(grid_for(n8, 256, ew_cap())), dim3(256), 0, stream,
                       reinterpret_cast<const T*>(x.data_ptr()), reinterpret_cast<T*>(y.data_ptr()), n8, (int)approx))
}

static void colsum_impl(const torch::Tensor& a, const torch::Tensor* x, torch::Tensor* out, torch::Tensor& dst,
                        int approx, int mode) {
  const int N = a.size(0), F = a.size(1);
  TORCH_CHECK(F % 8 == 0, "column count must be a multiple of 8");
  TORCH_CHECK(dst.scalar_type() == torch::kFloat32 && dst.numel() == F && dst.is_contiguous());
  if (N == 0) return;
  const int ctiles = (F + 511) / 512;
  int R = std::max(1, std::min(N / 16, ew_cap() / ctiles));
  const bool nt = ew_nt();
  auto part = torch::empty({R, F}, a.options().dtype(torch::kFloat32));
  auto stream = at::hip::getCurrentHIPStream();
  FOR_FLOAT_TYPES(a.scalar_type(), T, {
    const T* ap = reinterpret_cast<const T*>(a.data_ptr());
    const T* xp = x ? reinterpret_cast<const T*>(x->data_ptr()) : nullptr;
    T* op = out ? reinterpret_cast<T*>(out->data_ptr()) : nullptr;
    if (mode == 0)
      hipLaunchKernelGGL((nt ? rows_colsum_kernel<0, T, true> : rows_colsum_kernel<0, T, false>), dim3(ctiles, R), dim3(256), 0, stream, ap, xp, op,
                         part.data_ptr<float>(), N, F, approx);
    else
      hipLaunchKernelGGL((nt ? rows_colsum_kernel<1, T, true> : rows_colsum_kernel<1, T, false>), dim3(ctiles, R), dim3(256), 0, stream, ap, xp, op,
                         part.data_ptr<float>(), N, F, approx);
  })
  float* outs[1] = {dst.data_ptr<float>()};
  reduce_partials_auto(part, 1, R, F, outs, stream);
}

void gelu_bwd(torch::Tensor dy, torch::Tensor x, int64_t approx, c10::optional<torch::Tensor> dbias,
              torch::Tensor out) {
  check_vec8(dy);
  check_vec8(x);
  check_vec8(out);
  TORCH_CHECK(dy.scalar_type() == x.scalar_type() && out.scalar_type() == x.scalar_type());
  TORCH_CHECK(dy.numel() == x.numel() && out.numel() == x.numel());
  auto stream = at::hip::getCurrentHIPStream();
  if (dbias.has_value() && dbias->defined()) {
    TORCH_CHECK(x.dim() == 2, "fused bias gradient needs a 2-D input");
    colsum_impl(dy, &x, &out, *dbias, (int)approx, 1);
    return;
  }
  const int64_t n8 = x.numel() / 8;
  FOR_FLOAT_TYPES(x.scalar_type(), T,
    hipLaunchKernelGGL((ew_nt() ? gelu_bwd_kernel<T, true> : gelu_bwd_kernel<T, false>), dim3(grid_for(n8, 256, ew_cap())), dim3(256), 0, stream,
                       reinterpret_cast<const T*>(dy.data_ptr()), reinterpret_cast<const T*>(x.data_ptr()),
                       reinterpret_cast<T*>(out.data_ptr()), n8, (int)approx))
}

void colsum(torch::Tensor x, torch::Tensor out) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous() && x.dim() == 2);
  colsum_impl(x, nullptr, nullptr, out, 0, 0);
}

torch::Tensor gated_act_fwd(torch::Tensor g, torch::Tensor u, int64_t kind) {
  check_vec8(g);
  check_vec8(u);
  auto y = torch::empty_like(g);
  const int64_t n8 = g.numel() / 8;
  auto stream = at::hip::getCurrentHIPStream();
  FOR_FLOAT_TYPES(g.scalar_type(), T,
    hipLaunchKernelGGL((ew_nt() ? gated_fwd_kernel<T, true> : gated_fwd_kernel<T, false>), dim3(grid_for(n8, 256, ew_cap())), dim3(256), 0, stream,
                       reinterpret_cast<const T*>(g.data_ptr()), reinterpret_cast<const T*>(u.data_ptr()),
                       reinterpret_cast<T*>(y.data_ptr()), n8, (int)kind))
  return y;
}

torch::Tensor gated_act_packed(torch::Tensor gu, int64_t kind, c10::optional<torch::Tensor> out) {
  TORCH_CHECK(gu.is_cuda() && gu.is_contiguous() && gu.dim() == 2 && gu.size(1) % 16 == 0, "gu: [N, 2I], I % 8 == 0");
  TORCH_CHECK(reinterpret_cast<uintptr_t>(gu.data_ptr()) % 16 == 0);
  const int64_t N = gu.size(0), I = gu.size(1) / 2;
  torch::Tensor y;
  if (out.has_value() && out->defined()) {
    y = *out;
    TORCH_CHECK(y.is_contiguous() && y.numel() == N * I && y.scalar_type() == gu.scalar_type() &&
                    reinterpret_cast<uintptr_t>(y.data_ptr()) % 16 == 0,
                "gated_act_packed: out must be a contiguous 16-B aligned [N, I] tensor of gu's dtype");
  } else {
    y = torch::empty({N, I}, gu.options());
  }
  const int64_t n8 = N * I / 8;
  if (n8 == 0) return y;
  auto stream = at::hip::getCurrentHIPStream();
  FOR_FLOAT_TYPES(gu.scalar_type(), T,
    hipLaunchKernelGGL((ew_nt() ? gated_packed_kernel<T, true> : gated_packed_kernel<T, false>), dim3(grid_for(n8, 256, ew_cap())), dim3(256), 0, stream,
                       reinterpret_cast<const T*>(gu.data_ptr()), reinterpret_cast<T*>(y.data_ptr()), n8, (int)(I / 8),
                       (int)kind))
  return y;
}

std::vector<torch::Tensor> gated_act_bwd(torch::Tensor dy, torch::Tensor g, torch::Tensor u, int64_t kind) {
  check_vec8(dy);
  check_vec8(g);
  check_vec8(u);
  auto dg = torch::empty_like(g), du = torch::empty_like(u);
  const int64_t n8 = g.numel() / 8;
  auto stream = at::hip::getCurrentHIPStream();
  FOR_FLOAT_TYPES(g.scalar_type(), T,
    hipLaunchKernelGGL((ew_nt() ? gated_bwd_kernel<T, true> : gated_bwd_kernel<T, false>), dim3(grid_for(n8, 256, ew_cap())), dim3(256), 0, stream,
                       reinterpret_cast<const T*>(dy.data_ptr()), reinterpret_cast<const T*>(g.data_ptr()),
                       reinterpret_cast<const T*>(u.data_ptr()), reinterpret_cast<T*>(dg.data_ptr()),
                       reinterpret_cast<T*>(du.data_ptr()), n8, (int)kind))
  return {dg, du};
}

// dgu [N, 2I] (packed [d gate | d up]) from dy [N, I] and the packed forward input gu [N, 2I]
void gated_act_bwd_packed(torch::Tensor dy, torch::Tensor gu, torch::Tensor dgu, int64_t kind) {
  check_vec8(dy);
  check_vec8(gu);
  check_vec8(dgu);
  TORCH_CHECK(gu.dim() == 2 && gu.size(1) % 16 == 0 && dy.dim() == 2 && dy.size(0) == gu.size(0) &&
                  2 * dy.size(1) == gu.size(1) && dgu.sizes() == gu.sizes() && dy.scalar_type() == gu.scalar_type() &&
                  dgu.scalar_type() == gu.scalar_type(),
              "gated_act_bwd_packed: dy [N, I], gu / dgu [N, 2I], I % 8 == 0, one dtype");
  const int64_t I = dy.size(1), n8 = dy.numel() / 8;
  auto stream = at::hip::getCurrentHIPStream();
  FOR_FLOAT_TYPES(gu.scalar_type(), T,
    hipLaunchKernelGGL((ew_nt() ? gated_bwd_packed_kernel<T, true> : gated_bwd_packed_kernel<T, false>), dim3(grid_for(n8, 256, ew_cap())), dim3(256), 0, stream,
                       reinterpret_cast<const T*>(dy.data_ptr()), reinterpret_cast<const T*>(gu.data_ptr()),
                       reinterpret_cast<T*>(dgu.data_ptr()), n8, (int)(I / 8), (int)kind))
}

void embedding_fwd(torch::Tensor idx, torch::Tensor wte, torch::Tensor wpe, int64_t off, torch::Tensor out,
                   c10::optional<torch::Tensor> off_dev, double dropout_p, int64_t dropout_seed) {
  TORCH_CHECK(dropout_p >= 0.0 && dropout_p < 1.0, "dropout p must be in [0, 1)");
  TORCH_CHECK(idx.is_cuda() && idx.scalar_type() == torch::kInt64 && idx.dim() == 2);
  const int B = idx.size(0), T = idx.size(1), C = wte.size(1), V = wte.size(0);
  TORCH_CHECK(C % 8 == 0 && wpe.size(1) == C && wte.scalar_type() == wpe.scalar_type());
  const int64_t* od = nullptr;
  if (off_dev.has_value() && off_dev->defined()) {  // device offset: the caller bounds it (clamped here)
    TORCH_CHECK(off_dev->is_cuda() && off_dev->scalar_type() == torch::kInt64 && off_dev->numel() == 1);
    od = off_dev->data_ptr<int64_t>();
  } else {
    TORCH_CHECK(off + T <= wpe.size(0), "positions exceed the position table");
  }
  TORCH_CHECK(out.scalar_type() == torch::kFloat32 && out.numel() == (int64_t)B * T * C && out.is_contiguous());
  auto idxc = idx.contiguous();
  const int N = B * T;
  auto stream = at::hip::getCurrentHIPStream();
  FOR_FLOAT_TYPES(wte.scalar_type(), TW,
    hipLaunchKernelGGL(embed_fwd_kernel<TW>, dim3((N + 3) / 4), dim3(256), 0, stream, idxc.data_ptr<int64_t>(),
                       reinterpret_cast<const TW*>(wte.data_ptr()), reinterpret_cast<const TW*>(wpe.data_ptr()),
                       out.data_ptr<float>(), N, T, C, (int)off, V, od, (int)wpe.size(0), (uint64_t)dropout_seed,
                       (float)dropout_p))
}

void transpose_bf16_group(std::vector<torch::Tensor> ins, std::vector<torch::Tensor> outs) {
  TORCH_CHECK(ins.size() == outs.size(), "transpose_bf16: one output per input");
  auto stream = at::hip::getCurrentHIPStream();
  Transposes all{};
  int64_t tiles = 0;
  auto launch = [&] {
    if (all.n > 0)
      hipLaunchKernelGGL(transpose_bf16_kernel, dim3((unsigned)tiles), dim3(256), 0, stream, all);
    all.n = 0;
    tiles = 0;
  };
  for (size_t i = 0; i < ins.size(); ++i) {
    const torch::Tensor &in = ins[i], &out = outs[i];
    TORCH_CHECK(in.is_cuda() && out.is_cuda() && in.scalar_type() == torch::kBFloat16 &&
                    out.scalar_type() == torch::kBFloat16 && in.dim() == 2 && out.dim() == 2, "transpose_bf16: 2-D bf16");
    const int64_t R = in.size(0), C = in.size(1);
    TORCH_CHECK(in.is_contiguous() && out.is_contiguous() && out.size(0) == C && out.size(1) == R,
                "transpose_bf16: out must be the contiguous [C, R]");
    TORCH_CHECK(R % 64 == 0 && C % 64 == 0, "transpose_bf16: dims must be multiples of 64");
    if (R == 0 || C == 0) continue;
    const int64_t more = (R / 64) * (C / 64);
    if (all.n == kTransposes || tiles + more >= (int64_t)1 << 31) launch();
    all.m[all.n++] = Transpose{reinterpret_cast<const uint16_t*>(in.data_ptr()), reinterpret_cast<uint16_t*>(out.data_ptr()),
                               (int)R, (int)C, (int)tiles};
    tiles += more;
  }
  launch();
}

void transpose_bf16(torch::Tensor in, torch::Tensor out) { transpose_bf16_group({in}, {out}); }

void embedding_bwd(torch::Tensor dout, torch::Tensor idx, torch::Tensor dwte, torch::Tensor dwpe, int64_t off,
                   double dropout_p, int64_t dropout_seed) {
  TORCH_CHECK(dropout_p >= 0.0 && dropout_p < 1.0, "dropout p must be in [0, 1)");
  const int B = idx.size(0), T = idx.size(1), C = dwte.size(1), V = dwte.size(0);
  TORCH_CHECK(dout.scalar_type() == torch::kFloat32 && dwte.scalar_type() == torch::kFloat32 &&
              dwpe.scalar_type() == torch::kFloat32 && C % 4 == 0);
  TORCH_CHECK(off + T <= dwpe.size(0));
  auto idxc = idx.contiguous();
  const int N = B * T;
  auto stream = at::hip::getCurrentHIPStream();
  hipLaunchKernelGGL(embed_bwd_tok_kernel, dim3((N + 3) / 4), dim3(256), 0, stream, dout.data_ptr<float>(),
                     idxc.data_ptr<int64_t>(), dwte.data_ptr<float>(), N, C, V, (uint64_t)dropout_seed,
                     (float)dropout_p);
  hipLaunchKernelGGL(embed_bwd_pos_kernel, dim3(T), dim3(256), 0, stream, dout.data_ptr<float>(), dwpe.data_ptr<float>(),
                     B, T, C, (int)off, (uint64_t)dropout_seed, (float)dropout_p);
}

// cos / sin [T, n] fp32 for positions pos (device int64 [1]) + 0 .. T - 1 of inv_freq [n] (fp32)
std::vector<torch::Tensor> rope_table(torch::Tensor inv_freq, torch::Tensor pos, int64_t T) {
  TORCH_CHECK(inv_freq.is_cuda() && inv_freq.scalar_type() == torch::kFloat32 && inv_freq.dim() == 1 && inv_freq.is_contiguous(),
              "rope_table: fp32 inv_freq [n]");
  TORCH_CHECK(pos.is_cuda() && pos.scalar_type() == torch::kInt64 && pos.numel() == 1, "rope_table: int64 position [1] on the device");
  const int64_t n = inv_freq.numel();
  TORCH_CHECK(T >= 1 && n >= 1 && T * n < (int64_t)1 << 31, "rope_table: size");
  auto cosv = torch::empty({T, n}, inv_freq.options()), sinv = torch::empty({T, n}, inv_freq.options());
  hipLaunchKernelGGL(rope_table_kernel, dim3((unsigned)std::min<int64_t>(1024, (T * n + 255) / 256)), dim3(256), 0,
                     at::hip::getCurrentHIPStream(), inv_freq.data_ptr<float>(), pos.data_ptr<int64_t>(), cosv.data_ptr<float>(),
                     sinv.data_ptr<float>(), (int)T, (int)n);
  return {cosv, sinv};
}

// qkv's keys and values into the caches at pos (inv_freq given: q and k rotated); q [B, T, H, D], a view of qkv without rotation.
// None where it is not bf16 in rows of 16-byte pieces throughout.
c10::optional<torch::Tensor> prompt_kv(torch::Tensor qkv, c10::optional<torch::Tensor> inv_freq, torch::Tensor kc, torch::Tensor vc,
                                       int64_t pos, int64_t H, int64_t Hkv) {
  TORCH_CHECK(qkv.dim() == 3 && kc.dim() == 4 && kc.sizes() == vc.sizes() && H >= 1 && Hkv >= 1, "prompt_kv: shapes");
  const int64_t B = qkv.size(0), T = qkv.size(1), D = kc.size(3), cap = kc.size(2);
  TORCH_CHECK(qkv.size(2) == (H + 2 * Hkv) * D && kc.size(0) == B && kc.size(1) == Hkv && pos >= 0 && pos + T <= cap,
              "prompt_kv: sizes");
  auto aligned = [](const torch::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
  for (const auto* t : {&qkv, &kc, &vc})
    if (!(t->is_cuda() && t->get_device() == qkv.get_device() && t->scalar_type() == torch::kBFloat16 && t->is_contiguous() &&
          aligned(*t)))
      return c10::nullopt;
  const bool rope = inv_freq.has_value() && inv_freq->defined();
  if (D < 16 || D % 16 != 0 || D > 1024 || H + 2 * Hkv > 4096 || B * T < 1 || B * T > (int64_t)1 << 30 || pos + T > 1 << 24) return c10::nullopt;
  if (rope && !(inv_freq->is_cuda() && inv_freq->get_device() == qkv.get_device() && inv_freq->is_contiguous() &&
                inv_freq->dim() == 1 && inv_freq->numel() == D / 2 &&
                (inv_freq->scalar_type() == torch::kFloat32 || inv_freq->scalar_type() == torch::kBFloat16)))
    return c10::nullopt;
  auto q = rope ? torch::empty({B, T, H, D}, qkv.options())
                : qkv.as_strided({B, T, H, D}, {qkv.stride(0), qkv.stride(1), D, 1}, qkv.storage_offset());
  const int64_t items = rope ? (H + Hkv) * (D / 16) + Hkv * (D / 8) : 2 * Hkv * (D / 8);
  const int per_wg = (int)std::min<int64_t>(4, std::max<int64_t>(1, 256 / items));
  auto bp = [](const torch::Tensor& t) { return reinterpret_cast<__hip_bfloat16*>(t.data_ptr()); };
  auto launch = [&](auto kernel, auto* inv) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)((B * T + per_wg - 1) / per_wg)), dim3(256), rope ? per_wg * D * sizeof(float) : 0,
                       at::hip::getCurrentHIPStream(), bp(qkv), inv, bp(q), bp(kc), bp(vc), B * T, per_wg, (int)T, (int)H,
                       (int)Hkv, (int)D, cap, (int)pos);
  };
  if (!rope) launch(prompt_kv_kernel<false, float>, (const float*)nullptr);
  else if (inv_freq->scalar_type() == torch::kFloat32) launch(prompt_kv_kernel<true, float>, (const float*)inv_freq->data_ptr());
  else launch(prompt_kv_kernel<true, __hip_bfloat16>, (const __hip_bfloat16*)inv_freq->data_ptr());
  return q;
}

// out (optional): a preallocated contiguous tensor of qkv's shape and dtype (not aliasing qkv)
torch::Tensor rope_qkv(torch::Tensor qkv, torch::Tensor cosv, torch::Tensor sinv, int64_t H, int64_t Hkv, int64_t D,
                       bool inverse, c10::optional<torch::Tensor> out_opt) {
  TORCH_CHECK(qkv.is_cuda() && qkv.is_contiguous() && qkv.dim() == 3);
  const int64_t B = qkv.size(0), T = qkv.size(1);
  TORCH_CHECK(qkv.size(2) == (H + 2 * Hkv) * D && cosv.size(0) == T && cosv.size(1) == D / 2);
  torch::Tensor out;
  if (out_opt.has_value() && out_opt->defined()) {
    out = *out_opt;
    TORCH_CHECK(out.is_contiguous() && out.numel() == qkv.numel() && out.scalar_type() == qkv.scalar_type() &&
                    out.data_ptr() != qkv.data_ptr() && reinterpret_cast<uintptr_t>(out.data_ptr()) % 16 == 0,
                "rope_qkv: out must be a contiguous 16-B aligned tensor like qkv, not aliasing it");
    out = out.view(qkv.sizes());
  } else {
    out = torch::empty_like(qkv);
  }
  const int64_t rows = B * T;
  auto stream = at::hip::getCurrentHIPStream();
  const bool vec = D % 16 == 0 && cosv.is_contiguous() && sinv.is_contiguous() &&
                   cosv.scalar_type() == torch::kFloat32 && sinv.scalar_type() == torch::kFloat32 &&
                   reinterpret_cast<uintptr_t>(cosv.data_ptr()) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(sinv.data_ptr()) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(qkv.data_ptr()) % 16 == 0;
  if (vec) {
    const int64_t per = (H + Hkv) * (D / 16) + Hkv * D / 8;
    FOR_FLOAT_TYPES(qkv.scalar_type(), TT,
      hipLaunchKernelGGL(rope_vec_kernel<TT>, dim3(grid_for(rows * per)), dim3(256), 0, stream,
                         reinterpret_cast<const TT*>(qkv.data_ptr()), reinterpret_cast<TT*>(out.data_ptr()),
                         cosv.data_ptr<float>(), sinv.data_ptr<float>(), rows, (int)T, (int)H, (int)Hkv, (int)D,
                         inverse ? 1 : 0))
    return out;
  }
  FOR_FLOAT_TYPES(qkv.scalar_type(), TT,
    hipLaunchKernelGGL(rope_kernel<TT>, dim3(grid_for(rows * qkv.size(2))), dim3(256), 0, stream,
                       reinterpret_cast<const TT*>(qkv.data_ptr()), reinterpret_cast<TT*>(out.data_ptr()),
                       cosv.data_ptr<float>(), sinv.data_ptr<float>(), rows, (int)T, (int)H, (int)Hkv, (int)D,
                       inverse ? 1 : 0))
  return out;
}

void kv_quantize(torch::Tensor x, torch::Tensor q, torch::Tensor scale, int64_t pos) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous() && x.dim() == 4);
  const int B = x.size(0), T = x.size(1), Hkv = x.size(2), D = x.size(3);
  TORCH_CHECK(q.scalar_type() == torch::kInt8 && q.size(0) == B && q.size(1) == Hkv && q.size(3) == D);
  const int cap = q.size(2);
  TORCH_CHECK(pos + T <= cap, "cache overflow");
  const int rows = B * T * Hkv;
  auto stream = at::hip::getCurrentHIPStream();
  FOR_FLOAT_TYPES(x.scalar_type(), TT,
    hipLaunchKernelGGL(kv_quant_kernel<TT>, dim3((rows + 3) / 4), dim3(256), 0, stream,
                       reinterpret_cast<const TT*>(x.data_ptr()), q.data_ptr<int8_t>(), scale.data_ptr<float>(), B,
                       T, Hkv, D, cap, (int)pos))
}

std::vector<torch::Tensor> tensor_stats(torch::Tensor x, int64_t bins) {
  TORCH_CHECK(x.is_cuda() && x.is_contiguous());
  const int64_t n = x.numel();
  auto fopt = x.options().dtype(torch::kFloat32);
  if (n == 0) {
    auto z = torch::zeros({}, fopt);
    return {z, z, z, z, torch::zeros({bins}, fopt), torch::zeros({bins + 1}, fopt)};
  }
  const int G = grid_for(n, 256, 1024);
  auto p1 = torch::empty({G, 3}, fopt);
  auto stream = at::hip::getCurrentHIPStream();
  FOR_FLOAT_TYPES(x.scalar_type(), T,
    hipLaunchKernelGGL(stats_pass1_kernel<T>, dim3(G), dim3(256), 0, stream, reinterpret_cast<const T*>(x.data_ptr()),
                       n, p1.data_ptr<float>()))
  auto sum = p1.select(1, 0).to(torch::kFloat64).sum();
  auto mean = (sum / (double)n).to(torch::kFloat32);
  auto mn = p1.select(1, 1).min();
  auto mx = p1.select(1, 2).max();
  // torch.histogram widens an empty range by +-0.5 around a constant input
  auto same = mn.eq(mx);
  auto lo = torch::where(same, mn - 0.5f, mn);
  auto hi = torch::where(same, mx + 0.5f, mx);
  auto mmm = torch::stack({mean, lo, hi}).contiguous();
  auto p2 = torch::empty({G}, fopt);
  auto hist = torch::zeros({bins}, fopt);
  FOR_FLOAT_TYPES(x.scalar_type(), T,
    hipLaunchKernelGGL(stats_pass2_kernel<T>, dim3(G), dim3(256), bins * sizeof(float), stream,
                       reinterpret_cast<const T*>(x.data_ptr()), n, mmm.data_ptr<float>(), p2.data_ptr<float>(),
                       hist.data_ptr<float>(), (int)bins))
  auto var = p2.to(torch::kFloat64).sum() / (double)std::max<int64_t>(1, n - 1);
  auto stdv = var.sqrt().to(torch::kFloat32);
  auto edges = torch::linspace(0.0, 1.0, bins + 1, fopt) * (hi - lo) + lo;
  auto width = (hi - lo) / (double)bins;
  auto density = hist / ((double)n * width);
  return {mean, stdv, mn, mx, density, edges};
}

namespace penroz {
DeferredReduce& deferred_reduce() {
  static thread_local DeferredReduce d;
  return d;
}
}  // namespace penroz

// stream = 0: finish column reductions on the current stream (default)
void set_deferred_reduce_stream(int64_t stream, int64_t device) {
  penroz::deferred_reduce().stream = reinterpret_cast<hipStream_t>(stream);
  penroz::deferred_reduce().device = (int)device;
}

int64_t get_deferred_reduce_stream() { return reinterpret_cast<int64_t>(penroz::deferred_reduce().stream); }
