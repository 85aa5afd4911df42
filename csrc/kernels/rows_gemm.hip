// Linear layers of a few rows to a few thousand: out[M, N] = x[M, K] · W[N, K]ᵀ (+ bias), bf16 operands, fp32 sums, bf16 or fp32 out.
//
// Below products that fill the card with tiles of 256 lie the short steps: batches of up to 64 sequences, 256 training tokens,
// prompts of a few hundred rows. Their products need 1 to 5 us of memory or matrix time; what bounds them is how many bytes the
// card has on the way (about 1.1 us a trip, the ring's 96 KB per CU), so the tile is the smallest that one round of workgroups
// holds (rows_gemm_plan, host_plan.h). A workgroup of 4 waves owns 16×16 to 64×128 outputs; stages of 64 to 256 columns arrive by
// LDS-DMA in a ring (128-byte row pieces, whole cache lines, chunks permuted on the source side so that a fragment read covers all
// banks); the waves split the tile (WM × WN) or the columns of a stage (WK, added through LDS at the end, in order). Tiles that
// share weights run on one XCD. In order (WK = 1) a sum is one chain of MFMAs over k, as in the library's unsplit kernels, and from 32
// rows on bit for bit theirs up to K = 1024: training steps take that form there, where a rounding that falls otherwise changes every
// later layer's. With the columns split, 64 x 2048 x 2048 takes 6.1 us instead of 7.0. decode_gemm_acc adds to an fp32 residual in place (64 x 768 x
// 3072: 8.3 us in a kernel whose waves read their operands directly, 6.0 here). us, library / here (weights from memory): 64 x 768
// x 768 7.1 / 3.3, 64 x 2048 x 2048 8.9 / 6.1, 64 x 2048 x 6144 19.0 / 16.3 (32×32; 32×16 since: 13.3), 256 x 2304 x 768 7.7 / 6.5, 1024 x 1152 x 1024 9.7 / 9.2;
// at 16 rows, skinny_gemm / here: 768 x 768 9.7 / 3.3, 2048 x 2048 7.1 / 4.6, 7232 x 2048 12.3 / 8.2. A call costs the host 4 us, the
// library's 19. Tiles of 128×128 in rings of two to four stages were no faster than the library anywhere.
#include "common.h"
#include "host_plan.h"
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

namespace penroz {
namespace {

typedef __bf16 rg_bf16x8 __attribute__((ext_vector_type(8)));
typedef float rg_f32x4 __attribute__((ext_vector_type(4)));

// what becomes of a sum: it is the output, is added to it (fp32), or its gelu (erf form) is; kRgNarrow beside it: the output is
// not of 16-byte pieces
enum { kRgPlain = 0, kRgAdd = 1, kRgGelu = 2, kRgNarrow = 4 };

// glds16 of memory that nobody reads again soon
__device__ __forceinline__ void glds16_once(const void* g, unsigned lds_addr) {
  unsigned keep;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt\n\ts_mov_b32 m0, %0"
               : "=&s"(keep)
               : "v"(g), "s"(lds_addr)
               : "memory");
}

template <int P, int LEFT>
__device__ __forceinline__ void wait_stages(int left) {  // all but the newest `left` stages of P loads have landed
  if constexpr (LEFT > 0) {
    if (left >= LEFT) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LEFT * P) : "memory");
      return;
    }
    wait_stages<P, LEFT - 1>(left);
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
}

// ONCE: no cache keeps the weights (a kernel of its own: a choice between two loads costs the small products up to 0.4 us)
template <int FM, int FN, int WM, int WN, int WK, int KS, int NBUF, bool ONCE, typename OUT>
__global__ void __launch_bounds__(64 * WM * WN * WK) rows_gemm_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w,
                                                                      const bf16* __restrict__ bias, OUT* __restrict__ out, int M,
                                                                      int N, int K, int ldx, int ldw, int ldo, int tiles_m,
                                                                      int end) {
  constexpr int TM = 16 * FM * WM, TN = 16 * FN * WN, NW = WM * WN * WK;
  constexpr int SUB = (TM + TN) * 128, STAGE = WK * KS * SUB;  // a sub-slice of 64 columns: x rows, then W rows
  constexpr int COLS = 64 * WK * KS, PIECES = STAGE / 1024 / NW, PER_SUB = SUB / 1024;
  static_assert(STAGE % (1024 * NW) == 0 && (NBUF - 2) * PIECES <= 63 && NBUF >= 2, "ring geometry");
  static_assert(WK == 1 || WK * WM * WN * FM * FN * 1024 <= NBUF * STAGE, "the waves' sums fit the ring");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int nwg = gridDim.x, wg = blockIdx.x;
  const int xcd = wg & 7, qd = nwg >> 3, rd = nwg & 7;
  const int id = (xcd < rd ? xcd * (qd + 1) : rd * (qd + 1) + (xcd - rd) * qd) + (wg >> 3);
  const int tn = id / tiles_m, tm = id - tn * tiles_m;
  const int m0 = tm * TM, n0 = tn * TN;
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wk = wv / (WM * WN), wm = wv / WN % WM, wn = wv % WN;

  // piece p of a stage: 8 rows of a sub-slice; lane -> row (lane >> 3), 16-byte chunk (lane & 7) ^ swizzle
  const char* src[PIECES];
  int kofs[PIECES];
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const int p = wv * PIECES + i, sub = p / PER_SUB, row = (p % PER_SUB) * 8 + (lane >> 3);
    const int ch = (lane & 7) ^ ((row >> 1) & 7);
    kofs[i] = 64 * sub + 8 * ch;
    const bf16* r = row < TM ? x + (size_t)min(m0 + row, M - 1) * ldx : w + (size_t)min(n0 + row - TM, N - 1) * ldw;
    src[i] = reinterpret_cast<const char*>(r + kofs[i]);
  }
  const unsigned lds = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lds_void_t*)smem + wv * PIECES * 1024);
  const char* zero = reinterpret_cast<const char*>(g_zero16);
  auto dma = [&](int st, int buf) {
    const int k0 = st * COLS;
    if (k0 + COLS <= K) {
#pragma unroll
      for (int i = 0; i < PIECES; ++i) {
        if (!ONCE || (wv * PIECES + i) % PER_SUB * 8 < TM) glds16(src[i] + (size_t)k0 * 2, lds + buf * STAGE + i * 1024);
        else glds16_once(src[i] + (size_t)k0 * 2, lds + buf * STAGE + i * 1024);
      }
    } else {
#pragma unroll
      for (int i = 0; i < PIECES; ++i)
        glds16(k0 + kofs[i] < K ? src[i] + (size_t)k0 * 2 : zero, lds + buf * STAGE + i * 1024);
    }
  };

  const int r16 = lane & 15, kq = lane >> 4;
  auto frag = [&](const char* t, int row, int ch) {
    return *reinterpret_cast<const uint4*>(t + row * 128 + ((ch ^ ((row >> 1) & 7)) << 4));
  };
  rg_f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = rg_f32x4{0.f, 0.f, 0.f, 0.f};

  const int nst = (K + COLS - 1) / COLS;
#pragma unroll
  for (int t = 0; t < NBUF - 1; ++t)
    if (t < nst) dma(t, t);
  wait_stages<PIECES, NBUF - 2>(nst - 1);
  __syncthreads();
  int buf = 0;
  for (int st = 0; st < nst; ++st) {
    if (st + NBUF - 1 < nst) dma(st + NBUF - 1, buf == 0 ? NBUF - 1 : buf - 1);  // freed by the barrier of the step before
#pragma unroll
    for (int s = 0; s < 2 * KS; ++s) {
      const char* xt = smem + buf * STAGE + (wk * KS + (s >> 1)) * SUB;
      const char* wt = xt + TM * 128;
      uint4 a[FM], b[FN];
#pragma unroll
      for (int j = 0; j < FN; ++j) b[j] = frag(wt, 16 * (FN * wn + j) + r16, 4 * (s & 1) + kq);
#pragma unroll
      for (int i = 0; i < FM; ++i) a[i] = frag(xt, 16 * (FM * wm + i) + r16, 4 * (s & 1) + kq);
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(rg_bf16x8, b[j]),
                                                              __builtin_bit_cast(rg_bf16x8, a[i]), acc[i][j], 0, 0, 0);
    }
    if (st + 1 < nst) wait_stages<PIECES, NBUF - 2>(nst - 2 - st);
    __syncthreads();
    buf = buf + 1 == NBUF ? 0 : buf + 1;
  }
  const bool wide = (ldo & 3) == 0 && !(end & kRgNarrow);
  end &= ~kRgNarrow;
  // a lane holds row m = r16 of a block, columns 4·kq .. + 3
  auto store = [&](int i, int j, rg_f32x4 v) {
    const int m = m0 + 16 * (FM * wm + i) + r16, n = n0 + 16 * (FN * wn + j) + 4 * kq;
    if (m >= M || n >= N) return;
    OUT* o = out + (size_t)m * ldo + n;
    const int cnt = min(4, N - n);
    if (bias != nullptr)
      for (int r = 0; r < cnt; ++r) v[r] += to_f(bias[n + r]);
    if (end == kRgGelu)  // of the value as it is without the activation
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = gelu_f(to_f(from_f<OUT>(v[r])), 0);
    if (cnt == 4 && wide) {
      if constexpr (sizeof(OUT) == 2) {
        bf16 h[4] = {from_f<bf16>(v[0]), from_f<bf16>(v[1]), from_f<bf16>(v[2]), from_f<bf16>(v[3])};
        *reinterpret_cast<uint2*>(o) = *reinterpret_cast<const uint2*>(h);
      } else {
        float4* f = reinterpret_cast<float4*>(o);
        float4 c = end == kRgAdd ? *f : float4{0.f, 0.f, 0.f, 0.f};
        *f = float4{c.x + v[0], c.y + v[1], c.z + v[2], c.w + v[3]};
      }
    } else {
      for (int r = 0; r < cnt; ++r) o[r] = from_f<OUT>(end == kRgAdd ? to_f(o[r]) + v[r] : v[r]);
    }
  };
  if constexpr (WK == 1) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) store(i, j, acc[i][j]);
  } else {
    // every wave leaves its sums; the blocks, shared out over the waves, are added over the WK slices
    rg_f32x4* red = reinterpret_cast<rg_f32x4*>(smem);
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) red[(wv * FM * FN + i * FN + j) * 64 + lane] = acc[i][j];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        if ((i * FN + j) % WK != wk) continue;
        rg_f32x4 v = rg_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < WK; ++k) v += red[((k * WM * WN + wm * WN + wn) * FM * FN + i * FN + j) * 64 + lane];
        store(i, j, v);
      }
  }
}

}  // namespace
}  // namespace penroz

using namespace penroz;

static void rg_launch(int tile, bool in_order, const torch::Tensor& x, const torch::Tensor& w, const bf16* bias,
                      const torch::Tensor& out, int end, bool past) {
  const int64_t M = x.size(0), N = w.size(0), K = x.size(1);
  auto stream = at::hip::getCurrentHIPStream();
  // past: nothing holds the weights from one call to the next (past_caches, ops/gemm.py). Of 16 MB and more, each read by one workgroup,
  // they pass the caches then, which keep the smaller ones of a decode step. us, from memory, kept / not: 16 x 8192 x 2048 9.1 / 8.1, 16 x
  // 7232 x 2048 8.3 / 7.6, 16 x 12288 x 2048 14.0 / 12.8, 16 x 32768 x 1024 16.7 / 13.8; of 4 to 8 MB 2 % or nothing. Zozenex large, 16 rows,
  // 32 tokens 46.4 / 44.8 ms (with rows_gemm_low's tile). Weights that the caches hold come from there sooner: 32 x 8192 x 2048 14.9 / 19.7, 32 x 4096 x
  // 2048, 117 MB in all, 6.6 / 7.6, 9 x 32768 x 2048 26.6 / 29.6.
  const bool once = past && N * K >= (int64_t)8 << 20;
  auto launch = [&](auto kern, auto kern_once, int threads, int lds, int TM, int TN, auto* o) {
    const int64_t tiles_m = (M + TM - 1) / TM, tiles = tiles_m * ((N + TN - 1) / TN);
    if (once && tiles_m == 1) kern = kern_once;
    hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(threads), lds, stream, reinterpret_cast<const bf16*>(x.data_ptr()),
                       reinterpret_cast<const bf16*>(w.data_ptr()), bias, o, (int)M, (int)N, (int)K, (int)x.stride(0),
                       (int)w.stride(0), (int)out.stride(0), (int)tiles_m, end);
  };
#define PENROZ_RG(FM, FN, WM, WN, WK, KS, NB)                                                                    \
  launch(rows_gemm_kernel<FM, FN, WM, WN, WK, KS, NB, false, OUT>, rows_gemm_kernel<FM, FN, WM, WN, WK, KS, NB, true, OUT>, \
         64 * WM * WN * WK, NB * WK * KS * 128 * 16 * (FM * WM + FN * WN), 16 * FM * WM, 16 * FN * WN, o)
  auto typed = [&](auto* o) {
    using OUT = std::remove_pointer_t<decltype(o)>;
    if (tile == 6) PENROZ_RG(1, 1, 1, 1, 4, 1, 6);
    else if (tile == 1 && in_order) PENROZ_RG(1, 1, 2, 2, 1, 2, 4);
    else if (tile == 1 && rows_gemm_narrow(M, N)) PENROZ_RG(2, 1, 1, 1, 4, 1, 6);
    else if (tile == 1) PENROZ_RG(2, 2, 1, 1, 4, 1, 4);
    else if (tile == 2) PENROZ_RG(2, 4, 1, 1, 4, 1, 3);
    else if (tile == 3) PENROZ_RG(2, 2, 2, 2, 1, 2, 4);
    else if (tile == 4) PENROZ_RG(2, 2, 2, 2, 1, 2, 2);
    else if (!in_order && rows_gemm_low(M, N, K)) PENROZ_RG(1, 4, 1, 1, 4, 1, 2);
    else PENROZ_RG(2, 4, 2, 2, 1, 1, 3);
  };
#undef PENROZ_RG
  if (out.scalar_type() == torch::kFloat32) typed(out.data_ptr<float>());
  else typed(reinterpret_cast<bf16*>(out.data_ptr()));
}

// x · wᵀ (+ bias) into out, or (none given) into a new tensor, fp32 or of x's type; in_order: each sum in one chain over k; gelu: its
// gelu (erf form); past: rg_launch. None where rows_gemm_plan leaves the product to the library or a row is not of 16-byte pieces.
c10::optional<torch::Tensor> rows_gemm(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias,
                                       c10::optional<torch::Tensor> out_opt, bool fp32, bool in_order, bool gelu, bool past) {
  const bool given = out_opt.has_value() && out_opt->defined(), has_bias = bias.has_value() && bias->defined();
  if (!(x.is_cuda() && w.is_cuda() && x.get_device() == w.get_device() && x.scalar_type() == torch::kBFloat16 &&
        w.scalar_type() == torch::kBFloat16 && x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1)))
    return c10::nullopt;
  const int64_t M = x.size(0), N = w.size(0), K = x.size(1);
  auto rows_ok = [&](const torch::Tensor& t) {
    return t.stride(1) == 1 && t.stride(0) >= K && t.stride(0) % 8 == 0 && t.stride(0) < (int64_t)1 << 30 &&
           reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  const int tile = rows_gemm_plan(M, N, K, in_order);
  if (tile == 0 || !rows_ok(x) || !rows_ok(w)) return c10::nullopt;
  if (has_bias && !(bias->is_cuda() && bias->get_device() == x.get_device() && bias->scalar_type() == torch::kBFloat16 &&
                    bias->is_contiguous() && bias->numel() == N))
    return c10::nullopt;
  if (given) {
    const torch::Tensor& o = *out_opt;
    if (!(o.is_cuda() && o.get_device() == x.get_device() && o.scalar_type() == (fp32 ? torch::kFloat32 : torch::kBFloat16) &&
          o.dim() == 2 && o.size(0) == M && o.size(1) == N && o.stride(1) == 1 && o.stride(0) >= N && o.stride(0) < (int64_t)1 << 30 &&
          (o.stride(0) % 4 != 0 || reinterpret_cast<uintptr_t>(o.data_ptr()) % (4 * o.element_size()) == 0)))
      return c10::nullopt;
  }
  torch::Tensor out = given ? *out_opt : torch::empty({M, N}, x.options().dtype(fp32 ? torch::kFloat32 : torch::kBFloat16));
  const bf16* bp = has_bias ? reinterpret_cast<const bf16*>(bias->data_ptr()) : nullptr;
  rg_launch(tile, in_order, x, w, bp, out, gelu ? kRgGelu : kRgPlain, past);
  return out;
}

int64_t rows_gemm_tile(int64_t M, int64_t N, int64_t K, bool in_order) { return rows_gemm_plan(M, N, K, in_order); }

// decode_linear.hip
void gemv_add(const bf16* x, int64_t x_rs, const bf16* w, const bf16* bias, float* resid, int M, int N, int K, bool past);

// resid[M, N] += x · wᵀ + bias (fp32 residual, in place); up to 4 rows by decode_gemv's kernel (768 x 768 3.3 us here, 2.1 to 2.4 there)
void decode_gemm_acc(torch::Tensor x, torch::Tensor w, c10::optional<torch::Tensor> bias, torch::Tensor resid, bool past) {
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == torch::kBFloat16 && x.dim() == 2 && x.stride(1) == 1 &&
                  x.stride(0) % 8 == 0 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0,
              "decode_gemm_acc: bf16 x [M, K], rows 16-B aligned");
  const int64_t M = x.size(0), K = x.size(1);
  TORCH_CHECK(M >= 1 && K % 32 == 0, "decode_gemm_acc: K % 32 == 0");
  TORCH_CHECK(w.is_cuda() && w.scalar_type() == torch::kBFloat16 && w.dim() == 2 && w.is_contiguous() && w.size(1) == K &&
                  w.size(0) % 16 == 0 && reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
              "decode_gemm_acc: bf16 contiguous 16-B aligned W [N, K], N % 16 == 0");
  const int64_t N = w.size(0);
  TORCH_CHECK(resid.is_cuda() && resid.scalar_type() == torch::kFloat32 && resid.is_contiguous() && resid.dim() == 2 &&
                  resid.size(0) == M && resid.size(1) == N,
              "decode_gemm_acc: fp32 contiguous resid [M, N]");
  const bf16* bp = nullptr;
  if (bias.has_value() && bias->defined()) {
    TORCH_CHECK(bias->scalar_type() == torch::kBFloat16 && bias->is_contiguous() && bias->numel() == N,
                "decode_gemm_acc: bf16 bias [N]");
    bp = reinterpret_cast<const bf16*>(bias->data_ptr());
  }
  if (N == 0) return;
  if (K == 0) {  // gemv_add clamps its loads to a row's last piece
    if (bp != nullptr) resid.add_(*bias);
    return;
  }
  if (M <= 4 && K <= 8192 && N < 16384)
    return gemv_add(reinterpret_cast<const bf16*>(x.data_ptr()), x.stride(0), reinterpret_cast<const bf16*>(w.data_ptr()), bp,
                    resid.data_ptr<float>(), (int)M, (int)N, (int)K, past);
  if (x.stride(0) >= (int64_t)1 << 30) x = x.contiguous();  // the kernel takes strides of 32 bits
  const int tile = rows_gemm_plan(M, N, K, false);
  const bool narrow = reinterpret_cast<uintptr_t>(resid.data_ptr()) % 16 != 0;
  rg_launch(tile ? tile : 3, false, x, w, bp, resid, narrow ? kRgAdd | kRgNarrow : kRgAdd, past);
}
