// Wave and split counts of decode launches over a grid of shapes and workspace
// sizes: every plan fits its workspace and the kernel's limits, a split hint is
// followed, and a deterministic launch takes one plan in every workspace with
// room for it and one other below, whatever the size.  With an argument: reads
// shapes (batch, kv heads, group, head dim, blocks, format, scores) and prints
// each one's waves and splits, and the plain rule's.
#include <cstdio>
#include <vector>

#include "decode_plan.h"

using namespace tierkv;

int main(int argc, char**) {
  if (argc > 1) {
    int b, kv, g, d, nb, fmt, sc;
    while (std::scanf("%d %d %d %d %d %d %d", &b, &kv, &g, &d, &nb, &fmt, &sc) == 7) {
      const Plan p = plan_launch(b, kv * g, kv, nb, FBS, d, fmt, sc, 0, false, int64_t(1) << 50);
      std::printf("%d/%d %d/%d\n", p.nw, p.splits, g <= 8 ? 8 : 4, required_splits(int64_t(b) * kv, nb, g, 0));
    }
    return 0;
  }
  long long plans = 0, bad = 0, shapes = 0, two = 0;
  const int batches[] = {1, 2, 3, 7, 16, 31, 32, 40, 64, 65, 128, 1000};
  const int blocks[] = {1, 3, 8, 9, 31, 64, 95, 96, 129, 144, 256, 257, 400, 511, 512, 660, 1022, 1023, 1100, 2048, 5000};
  for (int batch : batches)
    for (int kv : {1, 4, 8, 16})
      for (int groups : {1, 3, 4, 8, 9, 16})
        for (int nb : blocks)
          for (int D : {64, 128})
            for (int sc = 0; sc < 2; ++sc)
              for (int hint : {0, 1, 3, 8}) {
                // The reference format's plan differs at head_dim 64 only.
                const int fmt = nb % 2 ? TIERKV_WARM_ABSMAX_I8 : TIERKV_WARM_REF_U8;
                const int heads = kv * groups;
                const int64_t units = int64_t(batch) * kv;
                auto bytes = [&](int s) { return ws_layout(batch, heads, kv, nb, FBS, D, sc, s).total; };
                const int64_t least = least_workspace(batch, heads, kv, nb, FBS, D, sc, hint);
                const int64_t full = bytes(reported_splits(units, nb, groups, hint));
                std::vector<int64_t> sizes = {least, least + 1, full - 1, full, full + 1, int64_t(1) << 50};
                for (int s : PLAN_SPLITS)
                  for (int d = -1; d <= 1; ++d) sizes.push_back(bytes(s) + d);
                auto plan = [&](bool det, int64_t ws) {
                  return plan_launch(batch, heads, kv, nb, FBS, D, fmt, sc, hint, det, ws);
                };
                const Plan big = plan(true, int64_t(1) << 50), small = plan(true, least);
                ++shapes;
                two += big.nw != small.nw || big.splits != small.splits;
                if (least > full || bytes(big.splits) > full) ++bad;
                for (int64_t ws : sizes) {
                  if (ws < least) continue;
                  for (int det = 0; det < 2; ++det) {
                    const Plan p = plan(det, ws);
                    ++plans;
                    const bool fits = bytes(p.splits) <= ws && p.splits >= 1 && p.splits >= std::min(nb, min_splits(nb)) &&
                                      (p.nw == 4 || (p.nw == 8 && groups <= 8)) &&
                                      (p.splits == 1 || p.splits <= nb) &&
                                      (hint == 0 || p.splits == required_splits(units, nb, groups, hint));
                    const Plan& want = bytes(big.splits) <= ws ? big : small;
                    const bool same = !det || (p.nw == want.nw && p.splits == want.splits);
                    if (!fits || !same) {
                      if (bad++ < 10)
                        std::printf("batch %d kv %d groups %d blocks %d D %d scores %d hint %d ws %lld det %d: %d waves "
                                    "%d splits\n", batch, kv, groups, nb, D, sc, hint, (long long)ws, det, p.nw, p.splits);
                    }
                  }
                }
              }
  for (int D : {64, 128})
    for (int fmt : {TIERKV_WARM_REF_U8, TIERKV_WARM_ABSMAX_I8})
      for (int sc = 0; sc < 2; ++sc) std::printf("waves %d %d %d %d\n", D, fmt, sc, waves_per_simd(D, fmt, sc));
  std::printf("static_lds %d\n", STATIC_LDS);
  // Workgroups a CU holds, by hand: eight heads of 64 dims with score sums in
  // LDS take 9.5 + 8 + 32 KB with four waves (three fit), 16 KB more with
  // eight; sixteen heads of 128 dims take 41.5 KB, and 89.5 with 48 KB of
  // statistics.
  const int abs = TIERKV_WARM_ABSMAX_I8;
  const int64_t got[] = {workgroups_per_cu(1024, 8, 64, abs, true, 4, 4), workgroups_per_cu(1024, 8, 64, abs, true, 8, 4),
                         workgroups_per_cu(256, 4, 64, abs, false, 4, 1), workgroups_per_cu(256, 4, 64, abs, false, 8, 1),
                         workgroups_per_cu(256, 4, 64, 0, false, 4, 1),   workgroups_per_cu(256, 4, 64, 0, false, 8, 1),
                         workgroups_per_cu(300, 16, 128, abs, false, 4, 1), workgroups_per_cu(384, 16, 128, abs, true, 4, 1),
                         workgroups_per_cu(384, 16, 64, abs, true, 4, 1), workgroups_per_cu(100, 4, 128, abs, false, 8, 1)};
  const int64_t want[] = {3, 1, 4, 2, 3, 1, 2, 1, 2, 1};
  for (size_t i = 0; i < sizeof(got) / sizeof(got[0]); ++i)
    if (got[i] != want[i]) {
      ++bad;
      std::printf("workgroups per CU %zu: %lld, not %lld\n", i, (long long)got[i], (long long)want[i]);
    }
  std::printf("shapes %lld (two plans %lld) plans %lld bad %lld\n", shapes, two, plans, bad);
  return bad != 0;
}
