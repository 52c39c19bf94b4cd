// Expansion of the embedding nets in one variable, shared by the host that
// builds it (expand.cpp) and the kernels that evaluate it (expand.hip).
//
// An embedding net maps one number per neighbour slot, s = (sw(r)/r - avg) /
// std, to L3 features, so for a given net G_f(s) = sum_k C[k][f] phi_k(x) with
// x a monotonic map of s onto [-1, 1] and phi_k polynomials of degree k; the
// nets are analytic, so |C[k]| falls geometrically and a few dozen terms
// reach the rounding level of fp64. The contraction of the environment rows
// then needs no per-slot feature at all:
//   T[m][f] = sum_slots R[m] G_f = sum_k C[k][f] M[m][k],
//   M[m][k] = sum_slots R[m] phi_k(x),
// one small product per (centre, section) instead of the net per slot, and
// in the backward (dM = C dT per centre and section)
//   sum_f dT[m][f] G_f  = sum_k dM[m][k] phi_k(x)   (and phi_k' for G_f').
//
// Variable: y = kExpandRmin sw(r)/r, z = 2 y / (1 + y), x = kExpandA z -
// kExpandB. It depends on the distance alone (avg and std of the pair enter
// the coefficients), so a slot's basis values serve every pair. y = 0 is the
// cutoff, y = 1 a distance of kExpandRmin; x reaches -1 a little below y = 0,
// because the derivative of a Chebyshev sum loses digits at the ends of its
// interval and most neighbours sit near the cutoff (error of G' at y <= 0.1, of the
// largest slope, seeded Cu / water / HEA nets: with the end at y = 0 2.1e-15 / 2.6e-14
// / 1.6e-14, with the margin 7.0e-16 / 7.2e-16 / 2.1e-15). z spends resolution
// where the neighbours are; against z = y it saves a tenth of the terms.
// Slots closer than kExpandRmin (shorter than any bond) evaluate the net
// itself.
//
// Basis: k = 64 h + 16 b + 4 p + l stands for T_64h(x) T_16b(x) T_4p(x) T_l(x)
// (T_n the Chebyshev polynomial; b, p, l in 0..3). It spans the same
// polynomials as T_0 .. T_k and needs a dozen values per slot; M is then a
// matrix product of (m, b) rows and (p, l) columns for the matrix cores.
// basis_values and basis_slopes are the kernels' evaluation of the factors (the
// host's check of the accuracy calls them too).
#pragma once

#include <hip/hip_runtime.h>

namespace dpamd {

constexpr double kExpandRmin = 0.6;              // A
constexpr double kExpandMargin = 1.0 / 32.0;
constexpr double kExpandA = 2.0 / (1.0 + kExpandMargin);
constexpr double kExpandB = (1.0 - kExpandMargin) / (1.0 + kExpandMargin);
constexpr int kExpandMaxTerms = 256;

// Sizes (in doubles) of one pair's coefficients in the operand order of the
// two products: forward B operand C[k = 4q + g][16 (2 u + e) + c] at
// ((q NU2 + u) 64 + lane) 2 + e, lane = 16 g + c; backward B operand
// C[16 t + c][f = 8 q + 2 g + e] at ((t NQ2 + q) 64 + lane) 2 + e, zero past L3.
constexpr int expand_nu2(int L3) { return ((L3 + 15) / 16 + 1) / 2; }
constexpr int expand_nq2(int L3) { return (L3 + 7) / 8; }
constexpr long expand_fwd_stride(int H, int L3) { return 16L * H * expand_nu2(L3) * 128; }
constexpr long expand_bwd_stride(int H, int L3) { return 4L * H * expand_nq2(L3) * 128; }

// Basis values T_1..T_3, T_4, T_8, T_12, T_16, T_32, T_48 (v[1..9], v[0] = 1),
// then T_64, T_128, T_192 for the groups in use.
template <int H>
constexpr int kNumBasis = 10 + (H > 1 ? 1 : 0) + (H > 2 ? 2 : 0);

template <int H>
__host__ __device__ __forceinline__ void basis_values(double x, double* v) {
  v[0] = 1.0;
  v[1] = x;
  v[2] = fma(2.0 * x, x, -1.0);
  v[3] = x * fma(4.0 * x, x, -3.0);
  v[4] = fma(2.0 * v[2], v[2], -1.0);
  v[5] = fma(2.0 * v[4], v[4], -1.0);
  v[6] = v[4] * fma(4.0 * v[4], v[4], -3.0);
  v[7] = fma(2.0 * v[5], v[5], -1.0);
  v[8] = fma(2.0 * v[7], v[7], -1.0);
  v[9] = v[7] * fma(4.0 * v[7], v[7], -3.0);
  if constexpr (H > 1) v[10] = fma(2.0 * v[8], v[8], -1.0);
  if constexpr (H > 2) {
    v[11] = fma(2.0 * v[10], v[10], -1.0);
    v[12] = v[10] * fma(4.0 * v[10], v[10], -3.0);
  }
}

// ... and their derivatives in x
template <int H>
__host__ __device__ __forceinline__ void basis_slopes(double x, const double* v, double* d) {
  d[0] = 0.0;
  d[1] = 1.0;
  d[2] = 4.0 * x;
  d[3] = fma(12.0 * x, x, -3.0);
  d[4] = 4.0 * v[2] * d[2];
  d[5] = 4.0 * v[4] * d[4];
  d[6] = fma(12.0 * v[4], v[4], -3.0) * d[4];
  d[7] = 4.0 * v[5] * d[5];
  d[8] = 4.0 * v[7] * d[7];
  d[9] = fma(12.0 * v[7], v[7], -3.0) * d[7];
  if constexpr (H > 1) d[10] = 4.0 * v[8] * d[8];
  if constexpr (H > 2) {
    d[11] = 4.0 * v[10] * d[10];
    d[12] = fma(12.0 * v[10], v[10], -3.0) * d[10];
  }
}

}  // namespace dpamd
