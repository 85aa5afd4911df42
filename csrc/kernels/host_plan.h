// Host-side launch planning shared by the HIP launch wrappers — plain C++ (no HIP headers), so
// the same code is also compiled into tests/native/host_plan_test.cpp and run under the host
// AddressSanitizer / UndefinedBehaviorSanitizer (tests/test_host_sanitizers.py).
#pragma once
#include <algorithm>
#include <cstdint>

namespace penroz {

struct SplitK {
  int splits;  // workgroups per output tile along K
  int klen;    // K range of one split (multiple of bk)
};

// Split-K count for the weight-gradient GEMM from a wave-quantisation cost model: the launch runs
// ceil(ntiles·s / slots) waves of workgroups, each 1/s of the K loop long, plus the fp32 slab
// round trip (s slabs written and read once) priced against the per-workgroup MFMA time.
// slots = resident workgroups (1 per CU for the 256-tile kernel, 2 for the 128-tile one).
inline SplitK plan_wgrad_splits(int M, int N, int K, int tile, int n_cu, int bk) {
  SplitK r{1, 0};
  if (M <= 0 || N <= 0 || K <= 0 || tile <= 0 || bk <= 0) return r;
  const int64_t tiles_m = (M + tile - 1) / tile, tiles_n = (N + tile - 1) / tile;
  const int64_t ntiles = tiles_m * tiles_n;
  const int64_t slots = tile == 256 ? std::max(1, n_cu) : 2 * (int64_t)std::max(1, n_cu);
  const double wg_full_k = (double)tile * tile * 2.0 * K / (tile == 256 ? 2.3e12 : 1.1e12);  // seconds
  double best = 1e30;
  const int smax = std::min(64, std::max(1, K / 512));
  for (int s = 1; s <= smax; ++s) {
    const double waves = (double)((ntiles * s + slots - 1) / slots);
    const double slab = s > 1 ? (double)s * M * N * 8.0 / 4.0e12 : 0.0;
    const double cost = waves * wg_full_k / s + slab;
    if (cost < best * 0.995) best = cost, r.splits = s;
  }
  const int64_t per = ((int64_t)K + r.splits - 1) / r.splits;
  r.klen = (int)((per + bk - 1) / bk * bk);
  r.splits = (int)(((int64_t)K + r.klen - 1) / r.klen);
  return r;
}

// Weight-gradient launch plan with a split TAIL: when the output tiles take more than one round of
// workgroups (one per CU) and the last round is mostly empty, the tiles of the full rounds run
// unsplit (direct read-add-write of the gradient, no slab) and only the last round's tiles are
// split along K, so that round is as full as the CUs allow and takes 1/tail_splits of a tile's
// time. GPT-2 lm_head (591 tiles): 2 + 1/3 rounds instead of 3 (or 5 half-rounds plus two
// full-size slabs). Falls back to the uniform plan above whenever that prices lower.
struct WgradPlan {
  int main_tiles;   // tiles [0, main_tiles): main_splits each
  int main_splits;  // 1 = direct into the gradient, > 1 = full-size fp32 slabs
  int main_klen;
  int tail_splits;  // tiles [main_tiles, ntiles): tail_splits each into per-tile slabs (0: none)
  int tail_klen;
};

inline WgradPlan plan_wgrad(int M, int N, int K, int tile, int n_cu, int bk) {
  const SplitK u = plan_wgrad_splits(M, N, K, tile, n_cu, bk);
  WgradPlan r{0, u.splits, u.klen, 0, 0};
  if (M <= 0 || N <= 0 || K <= 0 || tile != 256 || bk <= 0) {
    r.main_tiles = (M > 0 && N > 0 && tile > 0) ? (int)(((int64_t)(M + tile - 1) / tile) * ((N + tile - 1) / tile)) : 0;
    return r;
  }
  const int64_t ntiles = (int64_t)((M + tile - 1) / tile) * ((N + tile - 1) / tile);
  r.main_tiles = (int)ntiles;
  const int64_t slots = std::max(1, n_cu);
  if (ntiles <= slots) return r;
  const double wg_full_k = (double)tile * tile * 2.0 * K / 2.3e12;
  auto uniform_cost = [&](int s) {
    const double waves = (double)((ntiles * s + slots - 1) / slots);
    return waves * wg_full_k / s + (s > 1 ? (double)s * M * N * 8.0 / 4.0e12 : 0.0);
  };
  const int64_t rounds = (ntiles + slots - 1) / slots;
  const int64_t tail = ntiles - (rounds - 1) * slots;
  const int st = (int)std::min<int64_t>({64, slots / tail, std::max(1, K / 512)});
  if (st < 2) return r;
  const double tail_cost = (double)(rounds - 1) * wg_full_k + wg_full_k / st +
                           (double)tail * st * tile * tile * 8.0 / 4.0e12;
  if (tail_cost >= uniform_cost(u.splits) * 0.995) return r;
  r.main_tiles = (int)(ntiles - tail);
  r.main_splits = 1;
  r.main_klen = (int)(((int64_t)K + bk - 1) / bk * bk);
  const int64_t per = ((int64_t)K + st - 1) / st;
  r.tail_klen = (int)((per + bk - 1) / bk * bk);
  r.tail_splits = (int)(((int64_t)K + r.tail_klen - 1) / r.tail_klen);
  return r;
}

// Several weight gradients over the same K tokens: one launch of wgrad_group_kernel with tiles of tile_m × 128 (128 or 256), or
// each by the split kernel on its own (0). All estimates are fits (µs) to GPT-2's and Gemma-3 1B's layers, their heads and a
// layer of width 256 at 17 to 16384 tokens: a 32-token stage takes 0.43 with a card full of tiles (0.30 for one tile of 128 to a
// CU), 0.6 to 0.75 in the split kernel, which costs 20 whatever its size; outputs are written at 5.5 TB/s. Measured, one by one /
// together: GPT-2's layer 99 / 14 at 256 tokens, 134 / 62 at 3885, 275 / 243 at 16384; Gemma's 117 / 38, 302 / 239, 886 / 953; a
// head of 50304 x 768 119 / 104 at 1024, 176 / 189 at 2048; a layer of width 256 104 / 81 at 8192, 120 / 154 at 16384.
// shared: beside another stream's kernels a launch of several rounds holds every CU until its last round (Gemma-3 1B on two streams,
// 6 x 1024 tokens: 58.2 ms a step together, 55.8 one by one; GPT-2, whose layer is one round, 9.6 and 9.9). A single product is
// then the split kernel's, whose fewer workgroups leave the other stream CUs (Gemma-3 1B, each product as it comes, 1024 tokens:
// 24.6 ms a step with the grouped kernel, 22.4 with the split one; 1536 28.4 / 27.0, 2048 28.4 / 28.6).
inline int plan_wgrad_group(const int* M, const int* N, int n, int K, int n_cu, bool shared) {
  if (n <= 0 || K <= 0 || (shared && n == 1)) return 0;
  const double steps = (double)(((int64_t)K + 31) / 32);
  const int64_t cus = std::max(1, n_cu);
  double single = 0, store = 0;
  int64_t small = 0, large = 0;
  for (int i = 0; i < n; ++i) {
    if (M[i] <= 0 || N[i] <= 0) return 0;
    const int64_t tm = ((int64_t)M[i] + 127) / 128, tn = ((int64_t)N[i] + 127) / 128;
    small += tm * tn;
    large += (tm + 1) / 2 * tn;
    const double out = 4.0 * M[i] * N[i] / 5.5e6;
    store += out;
    const WgradPlan p = plan_wgrad(M[i], N[i], K, 256, n_cu, 32);
    const int64_t main = (int64_t)p.main_tiles * p.main_splits;
    single += 20 + (main > cus ? 0.75 : 0.6) * (double)((main + cus - 1) / cus) * p.main_klen / 32;
    if (p.tail_splits > 0) single += 0.75 * p.tail_klen / 32;
    single += p.main_splits > 1 ? 3 + 8.0 * p.main_splits * M[i] * N[i] / 20e6 : out;
  }
  const int64_t rest = small % (2 * cus);
  const double t128 = steps * (0.43 * (double)(small / (2 * cus)) + (rest > cus ? 0.43 : rest > 0 ? 0.30 : 0.0)) *
                      (1.0 + std::max(0, K - 4096) / 32768.0);  // operands from beyond the XCD's L2
  const double t256 = steps * 0.43 * (double)((large + cus - 1) / cus);
  if (std::min(t128, t256) + store + 6 >= single) return 0;
  const int tile = t128 <= t256 ? 128 : 256;
  if (shared && (tile == 128 ? small > 2 * cus : large > cus)) return 0;
  return tile;
}

// The tile of rows_gemm.hip for x [M, K] · W [N, K]ᵀ, or 0 for the library: the smallest tile that one round of workgroups on the
// MI355X's 256 CUs holds. 6: 16×16 and 1: 32×32 with the columns split over the waves (1 in order: two to a CU), 2: 32×64 with split
// columns, 3: 64×64, 4: 64×64 in a ring of two stages, two to a CU, 5: 64×128, two to a CU. Larger products are the library's, whose
// tiles of 256 read less. M x N x K, here / library, us:
//   * 6 64 x 768 x 3072 5.5 (1: 7.4) / 9.8, 16 x 2048 x 2048 4.6 (1: 5.7) / 8.1. One block beyond its round 1 is faster than two
//     rounds of it: 64 x 1152 x 6912 17.3 (6: 18.1) / 20.0, 64 x 1152 x 1024 4.3 (6: 5.6) / 8.4, 96 x 768 x 3072 7.3 (6: 9.3) /
//     7.6, 96 x 1152 x 6912 17.2 / 17.1 (32×32 each; rows_gemm_narrow's tile has these products now).
//   * 1 in order 256 x 1536 x 1024 5.8 / 8.6; 2 64 x 8192 x 2048 11.3 / 13.3, 256 x 1152 x 6912 23.9 / 24.2
//   * 3 beyond K = 2048 is 5 to 9 % slower than the library (256 x 12288 x 2048 35 / 27); 256 x 3072 x 2048 12.5 / 12.9, 400 x 1536 x
//     1152 8.0 / 9.6, but 400 x 2048 x 2048 11.9 / 11.0 and 1024 x 576 x 2048 11.9 / 10.5, at a fifth of its host time
//   * 4 and 5 only for K <= 1024, where their shorter rings do not wait: 512 x 2304 x 768 7.7 (4) / 8.5, 1024 x 3072 x 768
//     11.2 (5) / 11.4, 700 x 4096 x 1024 12.6 (5) / 11.8 (again a fifth of the host time), 2048 x 3072 x 768 18 (5) / 15.7
//   * 5 of up to 64 rows also to K = 2048: 64 x 32768 x 2048 35. Up to 8 rows those stay with skinny_gemm, so that the results of such
//     steps, a prompt of 8 sequences among them, keep their bits; rows_gemm_low's tile would be faster (5 x 32768 x 2048: skinny_gemm
//     32.0, 64×128 36.5, 16×64 27.1)
inline int rows_gemm_plan(int64_t M, int64_t N, int64_t K, bool in_order) {
  if (M <= 0 || N <= 0 || K <= 0 || K % 8 != 0 || M > 1 << 20 || N > 1 << 20 || K > 1 << 20) return 0;
  auto tiles = [&](int64_t tm, int64_t tn) { return ((M + tm - 1) / tm) * ((N + tn - 1) / tn); };
  if (!in_order && tiles(16, 16) <= 256) return 6;
  if (tiles(32, 32) <= (in_order ? 512 : 256)) return 1;
  if (!in_order && tiles(32, 64) <= 256) return 2;
  if (tiles(64, 64) <= 256 && K <= 2048) return 3;
  if (tiles(64, 64) <= 512 && K <= 1024) return 4;
  if ((tiles(64, 128) <= 384 && K <= 1024) || (M <= 64 && tiles(64, 128) <= 512 && K <= (M > 8 ? 2048 : 1024))) return 5;
  return 0;
}

// Tile 1 with split columns is 32×16 where one round holds that: the same sums in the same order, but more CUs, of which each takes
// some 22 B a cycle whatever the tile. us, 32×32 / 32×16, weights from memory, both in turn: 64 x 2048 x 6912 18.5 / 14.5, 64 x 2048 x
// 2048 7.1 / 6.4, 64 x 1152 x 6912 17.7 / 13.5, 64 x 1152 x 1024 4.9 / 4.6, 96 x 768 x 3072 9.2 / 7.5, 32 x 4096 x 2048 7.8 / 7.0, 256 x
// 512 x 2048 6.7 / 5.9, 65 x 832 x 768 4.1 / 3.8; of 256 columns the same (3.1). Two rounds of it are slower (64 x 3648 x 2048 7.7 / 11.3), and so is 16×8 in place of 16×16 (16 x 2048 x 2048 5.2 / 5.5).
inline bool rows_gemm_narrow(int64_t M, int64_t N) { return ((M + 31) / 32) * ((N + 15) / 16) <= 256; }

// Tile 5 of up to 16 rows, columns split, is 16×64, two workgroups to a CU and all of them at once: 64×128 brings 64 rows of x where 16
// are there, on one CU each. us, weights past the caches, 64×128 / 16×64, 16 rows: 16400 x 1152 13.7 / 11.8, 2048 23.9 / 17.6; 24576 x
// 1280 17.0 / 15.1, 2048 26.1 / 21.2; 32768 x 1152 15.9 / 15.8, 1536 20.4 / 19.1, 2048 33.1 / 26.8; but 32768 x 1024 14.6 / 14.7 and 50304 x
// 768 17.0 / 17.9, more than one round. (Narrower outputs of 1024 columns and fewer would gain too: 16400 x 1024 12.6 / 10.1.) 5 and 8 rows,
// skinny_gemm / 16×64: 16400 x 1280 17.8, 19.1 / 12.4, 2048 18.8, 19.8 / 17.5; 32768 x 1280 28.8, 30.9 / 16.6, 2048 32.0, 34.6 / 27.2; but
// 16400 x 1056 10.4, 11.0 / 12.4.
inline bool rows_gemm_low(int64_t M, int64_t N, int64_t K) { return M <= 16 && K > 1024 && N <= 32768; }

// Slices of the deterministic column reduction (reduce.h): ~sqrt(G) balances its two steps.
inline int reduce_slices(int G) {
  int s = 1;
  while ((int64_t)s * s < G) ++s;
  return s;
}

}  // namespace penroz
