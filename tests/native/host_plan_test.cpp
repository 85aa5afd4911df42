// Host-side unit test of the launch planners in csrc/kernels/host_plan.h, built and run by
// tests/test_host_sanitizers.py with -fsanitize=address,undefined (any report aborts the run).
#include "host_plan.h"

#include <cstdio>
#include <cstdlib>

using penroz::plan_wgrad_splits;

static int fails = 0;
#define EXPECT(c)                                                   \
  do {                                                              \
    if (!(c)) {                                                     \
      std::printf("FAIL %s:%d: %s\n", __FILE__, __LINE__, #c);      \
      ++fails;                                                      \
    }                                                               \
  } while (0)

int main() {
  // GPT-2 124M / XL weight-gradient shapes (K = tokens per step) and edge cases
  const int shapes[][3] = {{2304, 768, 65536}, {768, 768, 65536}, {3072, 768, 65536}, {768, 3072, 65536},
                           {50304, 768, 65536}, {50257, 768, 65536}, {4800, 1600, 65536}, {6400, 1600, 16384},
                           {8, 8, 1}, {200, 136, 1000}, {1, 1, 511}, {65536, 65536, 2147483647 / 2}};
  for (auto& s : shapes) {
    for (int tile : {128, 256}) {
      for (int bk : {32, 64}) {
        const auto p = plan_wgrad_splits(s[0], s[1], s[2], tile, 256, bk);
        EXPECT(p.splits >= 1 && p.splits <= 64);
        EXPECT(p.klen > 0 && p.klen % bk == 0);
        EXPECT((long long)p.klen * p.splits >= s[2]);              // covers K
        EXPECT((long long)p.klen * (p.splits - 1) < s[2]);         // no empty split
      }
    }
  }
  // split-tail plans: every tile covered once, the tail's splits cover K without an empty one
  const int tshapes[][3] = {{50304, 768, 65536}, {50257, 768, 65536}, {13824, 1152, 8192}, {262144, 1152, 8192},
                            {1152, 6912, 8192}, {6400, 1600, 16384}, {8, 8, 1}, {1 << 20, 768, 4096}};
  for (auto& s : tshapes) {
    const auto p = penroz::plan_wgrad(s[0], s[1], s[2], 256, 256, 32);
    const long long nt = (long long)((s[0] + 255) / 256) * ((s[1] + 255) / 256);
    EXPECT(p.main_tiles >= 0 && p.main_tiles <= nt);
    EXPECT(p.main_splits >= 1 && p.main_klen > 0 && p.main_klen % 32 == 0);
    EXPECT((long long)p.main_klen * p.main_splits >= s[2]);
    if (p.tail_splits > 0) {
      EXPECT(p.main_splits == 1 && p.main_tiles < nt && p.tail_splits >= 2);
      EXPECT(p.tail_klen % 32 == 0 && (long long)p.tail_klen * p.tail_splits >= s[2]);
      EXPECT((long long)p.tail_klen * (p.tail_splits - 1) < s[2]);
      EXPECT((nt - p.main_tiles) * p.tail_splits <= 256);  // the tail fits one round
    } else {
      EXPECT(p.main_tiles == nt);
    }
  }
  {  // GPT-2 lm_head: 591 tiles -> 512 direct + 79 tiles split 3 ways
    const auto p = penroz::plan_wgrad(50304, 768, 65536, 256, 256, 32);
    EXPECT(p.main_tiles == 512 && p.tail_splits == 3);
  }
  // degenerate inputs never divide by zero or overflow
  for (int bad : {0, -1}) {
    const auto p = plan_wgrad_splits(bad, 768, 1024, 256, 256, 64);
    EXPECT(p.splits == 1);
    const auto q = plan_wgrad_splits(768, 768, bad, 256, 0, 64);
    EXPECT(q.splits == 1);
    const auto w = penroz::plan_wgrad(768, bad, 1024, 256, 0, 32);
    EXPECT(w.tail_splits == 0 && w.main_splits >= 1);
  }
  for (int g : {0, 1, 2, 1024, 1 << 20, 2147483647}) {
    const int s = penroz::reduce_slices(g);
    EXPECT(s >= 1 && (long long)s * s >= g && (long long)(s - 1) * (s - 1) < (g > 1 ? g : 2));
  }
  // several weight gradients in one launch: a tile of 128 or 256 rows, or each by itself; any size, none of it overflowing
  const int gsizes[] = {-1, 0, 1, 8, 127, 128, 129, 768, 50304, 1 << 20, 1 << 30};
  for (int m : gsizes)
    for (int n : gsizes)
      for (int k : gsizes)
        for (int cus : {0, 1, 256})
          for (bool shared : {false, true}) {
            const int Ms[8] = {m, m, 768, m, 8, m, m, m}, Ns[8] = {n, 768, n, n, 8, n, n, n};
            for (int count : {0, 1, 2, 8}) {
              const int t = penroz::plan_wgrad_group(Ms, Ns, count, k, cus, shared);
              EXPECT(t == 0 || t == 128 || t == 256);
              if (count == 0 || k <= 0 || m <= 0 || n <= 0 || (shared && count == 1)) EXPECT(t == 0);
            }
          }
  {  // GPT-2's layer: together at every length up to 16384 tokens, beside a second stream as well; Gemma-3 1B's beside it never
    const int m[] = {768, 3072, 768, 2304}, n[] = {3072, 768, 768, 768};
    const int gm[] = {1152, 13824, 1152, 1536}, gn[] = {6912, 1152, 1024, 1152};
    for (int k : {1, 256, 3885, 16384}) {
      EXPECT(penroz::plan_wgrad_group(m, n, 4, k, 256, false) != 0 && penroz::plan_wgrad_group(m, n, 4, k, 256, true) != 0);
      EXPECT(penroz::plan_wgrad_group(gm, gn, 4, k, 256, true) == 0);
    }
    EXPECT(penroz::plan_wgrad_group(m, n, 4, 65536, 256, false) == 0);
  }
  // rows_gemm: a tile or the library; no size, odd column count or size beyond 2^20 has one, and every tile's grid fits its rule
  const int64_t rsizes[] = {-8, 0, 1, 8, 16, 17, 64, 65, 768, 772, 1024, 1152, 6912, 1 << 20, (1 << 20) + 8, (int64_t)1 << 40};
  for (int64_t m : rsizes)
    for (int64_t n : rsizes)
      for (int64_t k : rsizes)
        for (bool in_order : {false, true}) {
          const int t = penroz::rows_gemm_plan(m, n, k, in_order);
          EXPECT(t >= 0 && t <= 6);
          if (m <= 0 || n <= 0 || k <= 0 || k % 8 || m > 1 << 20 || n > 1 << 20 || k > 1 << 20) EXPECT(t == 0);
          if (in_order) EXPECT(t != 2 && t != 6);  // their waves split the columns
          const int64_t tm[] = {1, 32, 32, 64, 64, 64, 16}, tn[] = {1, 32, 64, 64, 64, 128, 16};
          if (t) EXPECT(((m + tm[t] - 1) / tm[t]) * ((n + tn[t] - 1) / tn[t]) <= 512);
        }
  // wide outputs of 9 to 16 rows of more than 1024 columns: the low tile in one round of 512 workgroups
  for (int64_t m : {4, 5, 8, 9, 16, 17, 64})
    for (int64_t n : {16384, 16385, 32768, 32769, 65536, 65537})
      for (int64_t k : {1024, 1032, 1272, 1280, 2048, 2056}) {
        const bool low = penroz::rows_gemm_low(m, n, k);
        EXPECT(low == (m <= 16 && n <= 32768 && k > 1024));
        if (low) EXPECT((n + 63) / 64 <= 512);
        if (n == 16384 || k == 1024) continue;
        const int want = k > 2048 || n > 65536 || m < 9 ? 0 : 5;
        EXPECT(penroz::rows_gemm_plan(m, n, k, false) == want);
        EXPECT(penroz::rows_gemm_plan(m, n, k, true) == want);
      }
  std::printf("host_plan_test: %s (%d failures)\n", fails ? "FAILED" : "ok", fails);
  return fails ? 1 : 0;
}
