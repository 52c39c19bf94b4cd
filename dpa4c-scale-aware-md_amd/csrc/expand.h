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
// interval and most neighbours sit near the cutoff (relative error of G' with
// the ends at y = 0: 1e-14; with the margin 5e-16). z spends resolution
// where the neighbours are; against z = y it saves a tenth of the terms.
// Slots closer than kExpandRmin (shorter than any bond) evaluate the net
// itself.
//
// Basis: k = 64 h + 16 b + 4 p + l stands for T_64h(x) T_16b(x) T_4p(x) T_l(x)
// (T_n the Chebyshev polynomial; b, p, l in 0..3). It spans the same
// polynomials as T_0 .. T_k and needs a dozen values per slot; M is then a
// matrix product of (m, b) rows and (p, l) columns for the matrix cores.
#pragma once

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

}  // namespace dpamd
