// Attention of several query rows per sequence over a bf16 key / value cache (prompts and continued portions of the
// decoders with a cache): causal, query row tq sits at position q_offset + tq.
//
// The rows of one KV head are (tq, head of its group), tq-major: a workgroup takes 64 of them, a wave 16, and goes
// over the cache in tiles of KT keys, so that a key or value is read once per 64 rows. (decode_kernel's workgroup per
// query row reads the whole cache for each.) us, decode_kernel / this one: 64 prompts of 64 tokens, 12 heads of 64
// 171 / 7.6, of 512 tokens 3220 / 114; one of 64 6.5 / 4.5, of 512 59 / 14.0; 4 query heads of 256 on one key head,
// 64 prompts of 100 tokens 171 / 16.9, 64 of 512 2366 / 113; 8 on 2 of 128, 4 prompts of 300 65 / 16.8; 8 of 512, 8 of 100
// 477 / 48.9. What bounds it: at few workgroups a tile's chain (load, barrier, scores, softmax, values: 1.2 us at D = 64,
// 2.3 at 256), at many the LDS reads of V and three products per weight.
//   * K and V tiles go through registers (the next tile's loads are on their way during this one's products) into
//     LDS, 16-byte chunks XOR-swizzled by row so that neither the row reads of K nor the column reads of V
//     (ds_read_b64_tr_b16) meet in a bank;
//   * scores are formed transposed, K times Qt with v_mfma_f32_16x16x32_bf16: a lane holds keys of ONE query row, the
//     softmax needs two exchanges across the wave per tile, and the weights are already the B operand of Vt times Pt;
//   * the weights are fp32 ones, every bit: they enter that product as three bf16 parts of 8 bits each. (As two parts, 16
//     bits, values that cancel leave 2^-18 of their size as an error instead of 2^-23; 64 prompts of 64 tokens 7.4 us, 64 of
//     512 102.)
//   * a value that is not finite would reach rows whose weight for it is zero (0 times inf): a tile that holds one is
//     multiplied on the vector unit, by the rows that see it.
// Where the row tiles leave CUs idle and the cache is long, the key tiles are split over workgroups and
// decode_combine_kernel adds the parts.
#include "common.h"
#include "prompt_attn.h"

namespace penroz {
namespace {

typedef __bf16 pa_bf16x8 __attribute__((ext_vector_type(8)));
typedef float pa_f32x4 __attribute__((ext_vector_type(4)));
typedef short pa_s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) pa_s16x4 pa_lds_s16x4;
typedef uint32_t pa_u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ pa_f32x4 pa_mfma(pa_u32x4 a, pa_u32x4 b, pa_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(pa_bf16x8, a), __builtin_bit_cast(pa_bf16x8, b), c,
                                                 0, 0, 0);
}

constexpr int kPaRows = 64;  // rows per workgroup, 16 per wave

// what the byte offset of a 16-byte chunk of a K row is XORed with: 16 consecutive rows' same chunk on 16 different
// slots of 256 bytes
template <int D> __device__ __forceinline__ int pa_kswz(int row) { return (D >= 128 ? row & 15 : (row >> 1) & 7) << 4; }
// of a V row: 8 consecutive rows' even chunk and the next one on 16 different slots
template <int D> __device__ __forceinline__ int pa_vswz(int row) { return (D >= 128 ? row & 7 : (row >> 1) & 3) << 5; }

template <int D, int KT>
__global__ void __launch_bounds__(256, D <= 256 ? 2 : 1) prompt_attn_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ kc, const bf16* __restrict__ vc, bf16* __restrict__ out,
    float* __restrict__ ws_o, float* __restrict__ ws_ml, int B, int Tq, int H, int Hkv, int cap, int q_offset,
    int row_tiles, int splits, float scale, int64_t q_rs) {
  constexpr int KS = D / 32, NT = D / 16, NB = KT / 16;
  constexpr int CH = D / 8, PT = KT * CH / 256;  // 16-byte chunks per row, per thread and tile
  constexpr int KB = KT * D * 2 > 4 * 16 * KT * 4 ? KT * D * 2 : 4 * 16 * KT * 4;
  __shared__ __attribute__((aligned(16))) char kt[KB];  // the K tile (and the weights of a tile with infinities)
  __shared__ __attribute__((aligned(16))) char vt[KT * D * 2];
  __shared__ uint32_t odd[4];  // by wave: V chunks with values that are not finite

  // sequences of one XCD by their heads (blocks 8 apart), the rows with the most keys first
  const int items = B * Hkv, items8 = (items + 7) / 8;
  const int xcd = blockIdx.x & 7;
  int id = blockIdx.x >> 3;
  const int split = id % splits;
  id /= splits;
  const int item = id % items8 * 8 + xcd, rt = row_tiles - 1 - id / items8;
  if (item >= items) return;
  const int g = item % Hkv, b = item / Hkv, G = H / Hkv;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int c16 = lane & 15, g4 = lane >> 4;

  const int rows = Tq * G, r0 = rt * kPaRows;
  const int row = min(r0 + 16 * w + c16, rows - 1);
  const bool live = r0 + 16 * w + c16 < rows;
  const int tq = row / G, head = g * G + (row - tq * G);
  const int limit = q_offset + tq;                                           // the row's last key
  const int wlast = q_offset + min(r0 + 16 * w + 15, rows - 1) / G;          // the wave's last key
  const int kend = q_offset + min(r0 + kPaRows - 1, rows - 1) / G + 1;       // keys that the workgroup sees
  const int tiles = (kend + KT - 1) / KT, per = (tiles + splits - 1) / splits;
  const int t0 = split * per, t1 = min(tiles, t0 + per);

  pa_u32x4 qf[KS];
  {
    const bf16* qp = q + ((size_t)b * Tq + tq) * q_rs + (size_t)head * D + 8 * g4;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[s] = *reinterpret_cast<const pa_u32x4*>(qp + 32 * s);
  }
  const size_t base = ((size_t)b * Hkv + g) * cap;
  pa_u32x4 kr[PT], vr[PT];
  auto load = [&](int k0) {
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int e = t + 256 * i, key = min(k0 + e / CH, kend - 1), ch = e % CH;
      kr[i] = *reinterpret_cast<const pa_u32x4*>(kc + (base + key) * D + 8 * ch);
      vr[i] = *reinterpret_cast<const pa_u32x4*>(vc + (base + key) * D + 8 * ch);
    }
  };
  constexpr bool AHEAD = D <= 256;  // (512 columns leave no registers for a tile on its way)
  if (AHEAD && t0 < t1) load(t0 * KT);

  const float c = scale * 1.4426950408889634f;
  float m = -INFINITY, l = 0.f;  // of this lane's row, the same in its four lanes
  pa_f32x4 o[NT];                // rows d = 16 i + 4 g4 + r of the output's column
#pragma unroll
  for (int i = 0; i < NT; ++i) o[i] = pa_f32x4{0.f, 0.f, 0.f, 0.f};

  for (int tile = t0; tile < t1; ++tile) {
    const int k0 = tile * KT;
    // (opaque: the offsets below are one XOR and add each, kept over the loop they are more registers than there are)
    int tt = t, kx = (g4 << 4) ^ pa_kswz<D>(c16), vx = pa_vswz<D>(4 * g4 + (c16 >> 2));
    asm volatile("" : "+v"(tt), "+v"(kx), "+v"(vx));
    if (tile > t0) __syncthreads();  // every wave is through with the last tile
    if (!AHEAD) load(k0);
    uint32_t bad = 0;
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int e = tt + 256 * i, r = e / CH, ch = e % CH;
      *reinterpret_cast<pa_u32x4*>(kt + r * (2 * D) + ((ch << 4) ^ pa_kswz<D>(r))) = kr[i];
      const pa_u32x4 v = k0 + r < kend ? vr[i] : pa_u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int j = 0; j < 4; ++j) bad |= (v[j] & 0x7f807f80u) + 0x00800080u;  // bit 15 / 31: all of the exponent set
      *reinterpret_cast<pa_u32x4*>(vt + r * (2 * D) + ((ch << 4) ^ pa_vswz<D>(r))) = v;
    }
    const bool any = __any((bad & 0x80008000u) != 0);
    if (lane == 0) odd[w] = any;
    __syncthreads();
    if (AHEAD && tile + 1 < t1) load(k0 + KT);
    const bool slow = (odd[0] | odd[1] | odd[2] | odd[3]) != 0;
    float p[NB][4];
    const bool sees = k0 <= wlast;  // (uniform over the wave)
    if (sees) {
      pa_f32x4 s[NB];
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        s[n] = pa_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < KS; ++i)
          s[n] = pa_mfma(*reinterpret_cast<const pa_u32x4*>(kt + (16 * n + c16) * (2 * D) + ((i << 6) ^ kx)), qf[i], s[n]);
      }
      float mx = -INFINITY;
#pragma unroll
      for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          p[n][r] = k0 + 16 * n + 4 * g4 + r <= limit ? s[n][r] * c : -INFINITY;
          mx = fmaxf(mx, p[n][r]);
        }
      mx = fmaxf(mx, lane_xor16(mx, g4 & 1));
      mx = fmaxf(mx, lane_xor32(mx, g4 >> 1));
      const float mn = fmaxf(m, mx), at = mn == -INFINITY ? 0.f : mn;  // (no score above -inf yet: nothing counts)
      const float alpha = m == -INFINITY ? 0.f : exp2f(m - mn);
      float sum = 0.f;
#pragma unroll
      for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          p[n][r] = exp2f(p[n][r] - at);
          sum += p[n][r];
        }
      sum += lane_xor16(sum, g4 & 1);
      sum += lane_xor32(sum, g4 >> 1);
      l = l * alpha + sum;
      m = mn;
#pragma unroll
      for (int i = 0; i < NT; ++i) o[i] *= alpha;
    }
    if (!slow) {
      if (sees) {
#pragma unroll
        for (int n = 0; n < NB; n += 2) {
          // k = 8 g4 + j of the product is key 16 n + 4 g4 + j (j < 4), 16 (n + 1) + 4 g4 + j - 4
          pa_u32x4 hi, mid, lo;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            float a = p[n + (j >> 1)][2 * (j & 1)], d = p[n + (j >> 1)][2 * (j & 1) + 1];
            hi[j] = pack_bf16x2(a, d);
            a -= __uint_as_float(hi[j] << 16), d -= __uint_as_float(hi[j] & 0xffff0000u);
            mid[j] = pack_bf16x2(a, d);
            a -= __uint_as_float(mid[j] << 16), d -= __uint_as_float(mid[j] & 0xffff0000u);
            lo[j] = pack_bf16x2(a, d);
          }
          const char* vp = vt + (16 * n + 4 * g4 + (c16 >> 2)) * (2 * D) + 8 * (lane & 3);
#pragma unroll
          for (int i = 0; i < NT; ++i) {
            const char* at = vp + ((i << 5) ^ vx);  // (16 rows on the swizzle is the same)
            const pa_s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pa_lds_s16x4*)at);
            const pa_s16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((pa_lds_s16x4*)(at + 16 * 2 * D));
            const uint2 ux = __builtin_bit_cast(uint2, x), uy = __builtin_bit_cast(uint2, y);
            const pa_u32x4 a = {ux.x, ux.y, uy.x, uy.y};
            o[i] = pa_mfma(a, hi, o[i]);
            o[i] = pa_mfma(a, mid, o[i]);
            o[i] = pa_mfma(a, lo, o[i]);
          }
        }
      }
    } else {
      __syncthreads();  // the scores of every wave are formed: the K tile gives way to the weights
      float* pw = reinterpret_cast<float*>(kt) + w * 16 * KT;  // [row][key]
      if (sees) {
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
          for (int r = 0; r < 4; ++r) pw[c16 * KT + 16 * n + 4 * g4 + r] = p[n][r];
      }
      __syncthreads();
      if (sees) {
        for (int key = 0; key < KT; ++key) {
          if (k0 + key > limit) break;
          const float pv = pw[c16 * KT + key];
#pragma unroll
          for (int i = 0; i < NT; ++i) {
            const int d = 16 * i + 4 * g4;
            const uint2 u = *reinterpret_cast<const uint2*>(vt + key * (2 * D) + ((2 * d) ^ pa_vswz<D>(key)));
            o[i][0] += pv * __uint_as_float(u.x << 16);
            o[i][1] += pv * __uint_as_float(u.x & 0xffff0000u);
            o[i][2] += pv * __uint_as_float(u.y << 16);
            o[i][3] += pv * __uint_as_float(u.y & 0xffff0000u);
          }
        }
      }
    }
  }
  if (!live) return;
  const size_t orow = ((size_t)b * Tq + tq) * H + head;
  if (splits == 1) {
    const float inv = l;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      float y[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = inv > 0.f ? o[i][r] / inv : 0.f;
      *reinterpret_cast<uint2*>(out + orow * D + 16 * i + 4 * g4) = uint2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
    }
    return;
  }
  const size_t wr = (size_t)split * B * Tq * H + orow;
#pragma unroll
  for (int i = 0; i < NT; ++i) *reinterpret_cast<pa_f32x4*>(ws_o + wr * D + 16 * i + 4 * g4) = o[i];
  if (g4 == 0) {
    ws_ml[2 * wr] = m;
    ws_ml[2 * wr + 1] = l;
  }
}

}  // namespace

// Where a round of decode_kernel's workgroups (a query row of a KV head each) or two hold all rows and the keys are few, a row on a
// CU of its own is sooner done than 64 together: with one head per KV head, and at 512 columns with more. us, decode_kernel / this
// one, 2 rows of 8 heads of 64 at 102 keys 4.7 / 5.8, 402 7.6 / 11.1, 1002 13.6 / 13.0; of 128 at 2 4.4 / 5.9, 102 5.8 / 8.6, 402
// 14.7 / 15.7, 1002 28.6 / 17.1; of 256 at 2 5.0 / 7.4, 202 14.5 / 20.6, 402 23.9 / 16.9; of 512 at 2 8.1 / 18.3, 202 54 / 70,
// 402 100 / 51. 280 to 512 workgroups: of 64 at 34 keys 5.0 / 4.5, 207 6.9 / 9.0; of 128 at 207 11.4 / 13.8, 404 24.2 / 16.4; of
// 256 at 57 7.7 / 9.8, 104 15.8 / 14.5; of 512 at 7 15.6 / 19.3, 34 30.6 / 28.1. 8 heads on 2: of 64 at 2 6.0 / 4.2, of 128
// 6.5 / 5.8, of 256 9.0 / 7.2, 102 15.6 / 13.8; of 512 at 2 13.8 / 18.4, 32 23.2 / 18.3. Gemma-3 1B's logits of 1 to 17 prompts of
// 9 to 500 tokens are 3.17 % off float64 with it, 3.18 % with decode_kernel (the bf16 residual's own error; 13 runs).
bool prompt_attn_applies(int64_t B, int64_t Tq, int64_t H, int64_t Hkv, int64_t D, int64_t keys) {
  if (Tq <= 1 || D < 64 || Hkv <= 0) return false;
  const int64_t G = H / Hkv, wgs = B * Hkv * Tq;
  if (G > 1) return !(D == 512 && wgs <= 256 && G * keys * D <= 40960);
  if (wgs <= 256) return keys * D > (D == 512 ? 122880 : 61440);
  if (wgs <= 512) return keys * D > (D == 512 ? 8192 : 32768) || (D == 64 && keys < 96);
  return true;
}

int prompt_attn_splits(int64_t items, int64_t rows, int64_t keys, int D, int part_keys) {
  // parts of 192 keys (128 of wide heads), as long as there are not two workgroups per CU without: a shorter part costs
  // more in its start and in the launch that adds the parts. 12 heads of 64, 4 rows at 1000 keys, one part / 512 / 256 /
  // 192 keys 22 / 16.3 / 14.0 / 12.2 us; 4 heads of 256, 16 rows at 900 keys, 4 sequences, 512 / 128 / 64 keys
  // 64 / 21.4 / 21.0; 2 rows at 4000 keys 44.7 / 28.2 / 38.7.
  const int64_t wgs = items * ((rows + kPaRows - 1) / kPaRows);
  const int64_t parts = part_keys > 0 ? (keys + part_keys - 1) / part_keys : keys / (D > 128 ? 128 : 192);
  return (int)std::max<int64_t>(1, std::min<int64_t>(512 / std::max<int64_t>(1, wgs), parts));
}

void prompt_attn_launch(const bf16* q, const bf16* kc, const bf16* vc, bf16* out, float* ws_o, float* ws_ml, int B,
                        int Tq, int H, int Hkv, int D, int cap, int q_offset, int splits, float scale, int64_t q_rs,
                        hipStream_t stream) {
  const int row_tiles = (Tq * (H / Hkv) + kPaRows - 1) / kPaRows;
  const dim3 grid((unsigned)((B * Hkv + 7) / 8 * 8 * row_tiles * splits));
  auto go = [&](auto d, auto kt) {
    hipLaunchKernelGGL((prompt_attn_kernel<decltype(d)::value, decltype(kt)::value>), grid, dim3(256), 0, stream, q, kc, vc,
                       out, ws_o, ws_ml, B, Tq, H, Hkv, cap, q_offset, row_tiles, splits, scale, q_rs);
  };
  using std::integral_constant;
  if (D == 64) go(integral_constant<int, 64>{}, integral_constant<int, 64>{});
  else if (D == 128) go(integral_constant<int, 128>{}, integral_constant<int, 64>{});
  else if (D == 256) go(integral_constant<int, 256>{}, integral_constant<int, 32>{});
  else go(integral_constant<int, 512>{}, integral_constant<int, 32>{});
}

}  // namespace penroz
