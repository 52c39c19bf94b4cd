// Splits of the general fitting chains' products and the workspace regions they
// write (host only).
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace dpamd {

// K slices for the first fitting layer: split only when the row blocks alone
// leave the device short of work, and keep at least 8 K chunks of 16 per
// slice. fp64: fewer than two blocks per compute unit (whole evaluation of
// 12,288 water atoms 798 us, against 823 with a target of four; 24,000 atoms
// 1,392 against 1,406; 3,993 and 98,304 atoms equal). fp32: fewer than four.
inline int fit_splits(int rows, int N, int K, int ncu, bool f32) {
  const int cols = N % 128 == 0 ? N / 128 : N % 80 == 0 ? N / 80 : N % 64 == 0 ? N / 64 : N / 16;
  const long blocks = (long)cols * ((rows + 63) / 64);
  const int nk = K / 16;
  int split = 1;
  while (blocks * split < (f32 ? 4L : 2L) * ncu && nk / (2 * split) >= 8) split *= 2;
  return split;
}

// Block shape of the fused dE/dD -> dE/dT kernels for a type of `rows` rows: eight
// waves (128 rows) when that gives every compute unit two blocks; four (64 rows)
// when it gives one; otherwise eight waves with the column groups split over
// blockIdx.y, enough ways to give every compute unit a block (at most one
// way per 16 groups a >= 16). Returns the split count; *waves the shape.
inline int ddt_shape(int rows, int L3, int ncu, int* waves) {
  const int nb8 = (rows + 127) / 128;
  *waves = 8;
  if (nb8 >= 2 * ncu) return 1;
  if (nb8 >= ncu) {
    *waves = 4;
    return 1;
  }
  const int smax = std::max(1, (L3 - 16) / 16);
  return std::min(smax, (ncu + nb8 - 1) / nb8);
}
inline int ddt_splits(int rows, int L3, int ncu) {
  int waves = 0;
  return ddt_shape(rows, L3, ncu, &waves);
}

// Per type the first layer's K slices [split][rows][F0] (elements of the nets'
// type, in one workspace of ws elements) and, on the fused kernels, their
// column-group partials [splits + 1][rows][64] (in one of dws doubles). The
// types' chains run concurrently: every split type has a region of its own, the
// others none. The slices take at most ws_max elements: the most slices any type
// has are halved until they do.
template <int NT>
struct FitPlan {
  int split[NT], dsplit[NT];
  size_t ws_at[NT], dws_at[NT];
  size_t ws = 0, dws = 0;
};

template <int NT>
FitPlan<NT> fit_plan(const int (&rows)[NT], int F0, int K, int L3, int ncu, bool f32, bool fused,
                     size_t ws_max = SIZE_MAX) {
  FitPlan<NT> p;
  for (int t = 0; t < NT; ++t) {
    p.split[t] = rows[t] > 0 ? fit_splits(rows[t], F0, K, ncu, f32) : 1;
    p.dsplit[t] = fused && rows[t] > 0 ? ddt_splits(rows[t], L3, ncu) : 1;
    p.dws_at[t] = p.dws;
    if (p.dsplit[t] > 1) p.dws += (size_t)(p.dsplit[t] + 1) * rows[t] * 64;
  }
  for (;;) {
    p.ws = 0;
    int most = 1;
    for (int t = 0; t < NT; ++t) {
      p.ws_at[t] = p.ws;
      if (p.split[t] > 1) p.ws += (size_t)p.split[t] * rows[t] * F0;
      most = std::max(most, p.split[t]);
    }
    if (p.ws <= ws_max || most == 1) return p;
    for (int t = 0; t < NT; ++t)
      if (p.split[t] == most) p.split[t] /= 2;
  }
}

}  // namespace dpamd
