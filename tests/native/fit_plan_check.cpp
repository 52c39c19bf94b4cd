// Workspace regions of the general fitting chains (csrc/fit_plan.h): over row
// counts per type on both sides of every rule, in every order, a split type's
// region must lie in the workspace and overlap no other's, and an unsplit type
// must take none; and with less memory than the slices ask for, they must fit it.
// Prints "ok" and the number of plans that mix split and unsplit types.
#include <cstdio>
#include <cstdlib>

#include "../../dpa4c-scale-aware-md_amd/csrc/fit_plan.h"

using namespace dpamd;

int main() {
  const int sizes[] = {0, 1, 64, 1000, 5440, 5441, 8192, 10880, 10881, 21760, 21761, 21888, 30000, 131072};
  constexpr int NT = 3, N = sizeof(sizes) / sizeof(sizes[0]);
  int mixed = 0;
  for (int k = 0; k < N * N * N; ++k)
    for (const bool f32 : {false, true})
      for (const bool fused : {false, true}) {
        const int rows[NT] = {sizes[k % N], sizes[k / N % N], sizes[k / N / N]};
        const FitPlan<NT> p = fit_plan(rows, 240, 1600, 100, 256, f32, fused);
        size_t ws = 0, dws = 0;
        int split = 0, whole = 0;
        for (int t = 0; t < NT; ++t) {
          const size_t n = (size_t)p.split[t] * rows[t] * 240, d = (size_t)(p.dsplit[t] + 1) * rows[t] * 64;
          if (p.split[t] > 1) {
            // (regions in type order: none below the end of the last)
            if (p.ws_at[t] < ws || p.ws_at[t] + n > p.ws) return std::printf("slices of type %d\n", t), 1;
            ws = p.ws_at[t] + n;
          }
          if (p.dsplit[t] > 1) {
            if (p.dws_at[t] < dws || p.dws_at[t] + d > p.dws) return std::printf("partials of type %d\n", t), 1;
            dws = p.dws_at[t] + d;
          }
          if (rows[t] > 0) p.split[t] > 1 ? ++split : ++whole;
        }
        if (ws != p.ws || dws != p.dws) return std::printf("unused memory\n"), 1;
        mixed += split > 0 && whole > 0;
        for (size_t most = p.ws; most > 0; most = most / 4 * 3) {
          const FitPlan<NT> q = fit_plan(rows, 240, 1600, 100, 256, f32, fused, most);
          bool less = q.dws == p.dws && q.ws <= most;
          size_t end = 0;
          for (int t = 0; t < NT; ++t) {
            less = less && q.split[t] >= 1 && q.split[t] <= p.split[t] && q.ws_at[t] >= end;
            if (q.split[t] > 1) end = q.ws_at[t] + (size_t)q.split[t] * rows[t] * 240;
          }
          if (!less || end > q.ws) return std::printf("slices in %zu elements\n", most), 1;
        }
      }
  std::printf("ok %d\n", mixed);
  return 0;
}
