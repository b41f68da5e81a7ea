// Host check of gemv_plan (eigen_amd/csrc/gemv.hip) over the matrices one
// launch takes (extent below 4 GB, both types and directions): the splits
// cover k, are at most 256 (a grid's y dimension ends at 65,536, and one
// thread adds a row's partial sums), and their partial sums fit the
// allocation-free entry's scratch; rows of A^T x that one load of a wave holds
// are not split, nor is Ax below 128 columns.  Built and run by tests/test_capi_cpu.py.
#include <cmath>
#include <cstdio>
#include <random>

#include "../eigen_amd/csrc/kernels.hpp"
#include "../include/eigen_amd.h"

int main() {
  std::mt19937_64 rng(1);
  auto log_uniform = [&](double hi) { return (int64_t)std::exp(std::uniform_real_distribution<>(0, std::log(hi))(rng)); };
  int64_t checked = 0;
  for (int es : {4, 8})
    for (int trans : {0, 1})
      for (int i = 0; i < 200000; ++i) {
        const int64_t room = 0xFFFFFFFFll / es - 64;
        int64_t m = log_uniform((double)room), k = log_uniform((double)room / (double)m);
        if (i == 0) m = 1, k = room;  // a dot product of the whole range
        if (i == 1) m = room, k = 1;
        if (i == 2) m = 4, k = 100000000;
        const eh::GemvPlan g = eh::gemv_plan(trans, (int)m, (int)k, es);
        const size_t ws = eh::gemv_workspace_bytes(g, (int)m, es);
        if (trans && k * es <= 1024 && (g.splits != 1 || g.batch != 8 || (int64_t)g.blocks * g.rows < m)) {
          std::printf("FAIL short rows es=%d m=%lld k=%lld: %d splits, batch %d\n", es, (long long)m, (long long)k, g.splits,
                      g.batch);
          return 1;
        }
        if (!trans && k < 128 && g.splits != 1) {
          std::printf("FAIL few columns es=%d m=%lld k=%lld: %d splits\n", es, (long long)m, (long long)k, g.splits);
          return 1;
        }
        if (g.blocks < 1 || g.splits < 1 || g.splits > 256 || (int64_t)g.per * g.splits < k ||
            (int64_t)g.per * (g.splits - 1) >= k || ws > EH_NOALLOC_SCRATCH_BYTES) {
          std::printf("FAIL trans=%d es=%d m=%lld k=%lld: %d splits of %d, %d blocks, %zu bytes\n", trans, es, (long long)m,
                      (long long)k, g.splits, g.per, g.blocks, ws);
          return 1;
        }
        ++checked;
      }
  // short columns share cache lines: never read with the non-temporal hint
  for (int m : {1, 50, 100, 250, 500, 4096}) {
    if (eh::gemv_streams(false, m, 1u << 30) != (m >= 500) || eh::gemv_streams(false, m, 1u << 27)) {
      std::printf("FAIL hint for Ax of %d rows\n", m);
      return 1;
    }
  }
  std::printf("ALL PASSED (%lld)\n", (long long)checked);
  return 0;
}
