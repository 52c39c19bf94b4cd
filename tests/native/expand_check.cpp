// The embedding nets' expansion on the host (csrc/expand.cpp): for each model
// file named on the command line, prints one line
//   ok H max|G - sum C phi| max|G' - sum C phi'| the same near the cutoff
//   max|G| max|G'| (differences of the two layouts)
// over distances from the range's end to the cutoff, with the coefficients
// read back from both operand layouts, the basis from the kernels' own functions
// in fp64 and the net and its tangent in extended precision; or "none"
// when some net has no short enough expansion. The best of three builds' times,
// in ms, goes to stderr, a line a model.
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <fstream>
#include <iterator>

#include "../../dpa4c-scale-aware-md_amd/csrc/expand.h"
#include "../../dpa4c-scale-aware-md_amd/csrc/model.h"

using namespace dpamd;
namespace dpamd {
bool emb_supported(int, int, int) { return true; }
}  // namespace dpamd
using ld = long double;

// the larger magnitude, NaN if either is
static double larger(double a, ld b) {
  const double v = std::fabs((double)b);
  return v <= a || std::isnan(a) ? a : v;
}

int main(int argc, char** argv) {
  for (int q = 1; q < argc; ++q) {
    std::ifstream in(argv[q], std::ios::binary);
    const std::vector<unsigned char> buf((std::istreambuf_iterator<char>(in)), {});
    ModelHost m;
    if (!parse_model(buf.data(), buf.size(), m).empty()) return 1;
    ExpandHost e;
    bool ok = false;
    double best = 1e30;
    for (int k = 0; k < 3; ++k) {
      const auto t0 = std::chrono::steady_clock::now();
      e = ExpandHost{};
      ok = build_expansion(m, e);
      const std::chrono::duration<double, std::milli> t = std::chrono::steady_clock::now() - t0;
      best = std::min(best, t.count());
    }
    std::fprintf(stderr, "%.3f\n", best);
    if (!ok) {
      std::printf("none\n");
      continue;
    }
    const int np = m.ntypes * m.ntypes, F = m.emb[2], N = 64 * e.H;
    const int NU2 = expand_nu2(F), NQ2 = expand_nq2(F);
    double eg = 0, ed = 0, en = 0, gm = 0, dm = 0;
    int layouts = 0;
    for (int p = 0; p < np; ++p) {
      const double* cf = e.fwd.data() + p * expand_fwd_stride(e.H, F);
      const double* cb = e.bwd.data() + p * expand_bwd_stride(e.H, F);
      std::vector<double> C((size_t)N * F);
      for (int k = 0; k < N; ++k)
        for (int f = 0; f < F; ++f) {
          const double v = cf[(((k / 4) * NU2 + f / 32) * 64 + 16 * (k % 4) + f % 16) * 2 + f / 16 % 2];
          const double w = cb[(((k / 16) * NQ2 + f / 8) * 64 + 16 * (f % 8 / 2) + k % 16) * 2 + f % 2];
          layouts += v != w || (k >= 16 * e.blocks[p] && v != 0.0);
          C[(size_t)k * F + f] = v;
        }
      const double avg = m.davg[4 * p], sd = m.dstd[4 * p];
      for (int s = 0; s <= 200; ++s) {
        const double y = s / 200.0;  // rmin sw / r: 0 at the cutoff, 1 at the range's end
        // basis functions and slopes as the kernels form them
        const double iv = 1.0 / (1.0 + y), x = fma(kExpandA * 2.0 * y, iv, -kExpandB);
        const int H = e.H;
        double v[kNumBasis<4>], sl[kNumBasis<4>];
        if (H == 1) basis_values<1>(x, v), basis_slopes<1>(x, v, sl);
        else if (H == 2) basis_values<2>(x, v), basis_slopes<2>(x, v, sl);
        else basis_values<4>(x, v), basis_slopes<4>(x, v, sl);
        double c[16], dc[16];
        for (int k = 0; k < 16; ++k) {
          const int l = k % 4, p4 = k / 4 ? 3 + k / 4 : 0;
          c[k] = v[l] * v[p4];
          dc[k] = fma(sl[l], v[p4], v[l] * sl[p4]);
        }
        // the net and its slope in extended precision
        std::vector<ld> h{((ld)y / (ld)kExpandRmin - avg) / sd}, t{1};
        const double* P = m.emb_params.data() + (size_t)p * m.emb_block;
        const int L[4] = {1, m.emb[0], m.emb[1], m.emb[2]};
        for (int k = 0; k < 3; ++k) {
          std::vector<ld> z(L[k + 1]), zt(L[k + 1]);
          for (int f = 0; f < L[k + 1]; ++f) {
            ld a = P[L[k] * L[k + 1] + f], at = 0;
            for (int c = 0; c < L[k]; ++c) {
              a += h[c] * P[c * L[k + 1] + f];
              at += t[c] * P[c * L[k + 1] + f];
            }
            z[f] = std::tanh(a);
            zt[f] = (1 - z[f] * z[f]) * at;
            if (k > 0 && L[k + 1] == 2 * L[k]) {
              z[f] += h[f % L[k]];
              zt[f] += t[f % L[k]];
            }
          }
          P += L[k] * L[k + 1] + L[k + 1];
          h = z;
          t = zt;
        }
        const double dxds = kExpandA * 2.0 * iv * iv * kExpandRmin * sd;
        for (int f = 0; f < F; ++f) {
          // (sums of 16 terms, then over the blocks, as the backward)
          double g = 0, d = 0;
          for (int k = 0; k < N; k += 16) {
            double Y = 0, Yd = 0;
            for (int q = 0; q < 16; ++q) {
              Y = fma(C[(size_t)(k + q) * F + f], c[q], Y);
              Yd = fma(C[(size_t)(k + q) * F + f], dc[q], Yd);
            }
            const int b = k / 16 % 4 ? 6 + k / 16 % 4 : 0, h64 = k / 64 ? 9 + k / 64 : 0;
            const double w = v[b] * v[h64], dw = fma(sl[b], v[h64], v[b] * sl[h64]);
            g = fma(w, Y, g);
            d = fma(dw, Y, fma(w, Yd, d));
          }
          eg = larger(eg, g - h[f]);
          ed = larger(ed, d * dxds - t[f]);
          gm = larger(gm, h[f]);
          dm = larger(dm, t[f]);
          if (y <= 0.1) en = larger(en, d * dxds - t[f]);
        }
      }
    }
    std::printf("ok %d %.3e %.3e %.3e %.3e %.3e %d\n", e.H, eg, ed, en, gm, dm, layouts);
  }
  return 0;
}
