// Host side of the embedding nets' expansion (expand.h): coefficients by
// Chebyshev interpolation in extended precision, their check, and the layouts
// the kernels read.
#include "expand.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <exception>
#include <thread>

#include "model.h"

namespace dpamd {

namespace {

using ld = long double;  // 64-bit significand: the coefficients' derivative
                         // amplifies their noise by k^2 near the cutoff

// One net at s, in extended precision (x, y: scratch of at least L3 values).
void net_ld(const ModelHost& m, const double* P, ld s, std::vector<ld>& x, std::vector<ld>& y) {
  const int L[4] = {1, m.emb[0], m.emb[1], m.emb[2]};
  x[0] = s;
  for (int k = 0; k < 3; ++k) {
    const int in = L[k], out = L[k + 1];
    const double* W = P;
    const double* b = P + (long)in * out;
    P = b + out;
    for (int f = 0; f < out; ++f) {
      // (two sums in registers: an extended-precision value in memory costs
      // several cycles a load and store)
      ld z0 = b[f], z1 = 0.0L;
      int q = 0;
      for (; q + 1 < in; q += 2) {
        z0 += x[q] * W[(long)q * out + f];
        z1 += x[q + 1] * W[(long)(q + 1) * out + f];
      }
      if (q < in) z0 += x[q] * W[(long)q * out + f];
      const ld t = std::tanh(z0 + z1);
      y[f] = t + (out == in && k > 0 ? x[f] : out == 2 * in && k > 0 ? x[f % in] : 0.0L);
    }
    std::swap(x, y);
  }
}

// c_0 .. c_{n-1} over T_k (stride F values) -> the same polynomial over
// T_{S b} T_a, a < S: T_{S b + a} = 2 T_{S b} T_a - T_{S b - a}.
void to_products(ld* c, int n, int S, int F) {
  for (int b = n / S - 1; b > 0; --b)
    for (int a = S - 1; a > 0; --a)
      for (int f = 0; f < F; ++f) {
        const ld v = c[(long)(b * S + a) * F + f];
        c[(long)(b * S + a) * F + f] = 2 * v;
        c[(long)(b * S - a) * F + f] -= v;
      }
}

// f(0) .. f(n - 1) over the host's cores (up to 8). What an f throws ends the
// others' work too and is thrown again once every thread has.
template <class Fn>
void parallel(int n, Fn&& f) {
  std::atomic<int> next{0};
  std::atomic<bool> failed{false};
  std::exception_ptr error;  // written by the thread that sets failed
  auto work = [&]() {
    try {
      for (int k = next++; k < n && !failed; k = next++) f(k);
    } catch (...) {
      if (!failed.exchange(true)) error = std::current_exception();
    }
  };
  std::vector<std::thread> pool;
  try {
    pool.reserve(7);
    for (int q = 1; q < std::min(n, 8); ++q) pool.emplace_back(work);
  } catch (const std::exception&) {
    // fewer threads than asked for: the rest of the work stays here
  }
  work();
  for (auto& t : pool) t.join();
  if (error) std::rethrow_exception(error);
}

// Chebyshev coefficients [n][L3] of the nets of `pairs` from n nodes (even),
// and per pair the number of terms (a multiple of 16, 0 if none will do) past
// which the magnitudes of every feature's coefficients sum to at most 2^-55
// of the largest feature: below the rounding of the sum itself, and small
// enough that the derivative's truncation stays below its rounding too.
void coefficients(const ModelHost& m, const std::vector<int>& pairs, int n,
                  std::vector<std::vector<ld>>& coef, std::vector<int>& terms) {
  const int np = (int)pairs.size(), F = m.emb[2];
  const ld pi = 3.14159265358979323846264338327950288L;
  std::vector<ld> cosine(4 * n);  // cos(i pi / 2n): exact angles for cos(k (2j + 1) pi / 2n)
  for (int i = 0; i < 4 * n; ++i) cosine[i] = std::cos((ld)i * pi / (2 * n));
  std::vector<ld> val((size_t)np * n * F);  // [pair][feature][node]
  for (int p : pairs) coef[p].assign((size_t)n * F, 0.0L);
  parallel(np * n, [&](int k) {
    const int p = pairs[k / n], j = k % n;
    const ld z = (cosine[2 * j + 1] + (ld)kExpandB) / (ld)kExpandA;
    const ld s = (z / (2 - z) / (ld)kExpandRmin - (ld)m.davg[(size_t)p * 4]) / (ld)m.dstd[(size_t)p * 4];
    std::vector<ld> x(F), y(F);
    net_ld(m, m.emb_params.data() + (size_t)p * m.emb_block, s, x, y);
    for (int f = 0; f < F; ++f) val[((size_t)(k / n) * F + f) * n + j] = x[f];
  });
  parallel(np * F, [&](int q) {
    const ld* v = val.data() + (size_t)q * n;
    ld* c = coef[pairs[q / F]].data() + q % F;
    // node n - 1 - j lies opposite node j: T_k there is (-1)^k T_k here
    std::vector<ld> fold(n);
    for (int j = 0; j < n / 2; ++j) {
      fold[j] = v[j] + v[n - 1 - j];
      fold[n / 2 + j] = v[j] - v[n - 1 - j];
    }
    for (int k = 0; k < n; ++k) {
      const ld* w = fold.data() + (k % 2 ? n / 2 : 0);
      ld sum = 0.0L;
      int at = k;  // k (2j + 1) mod 4n
      for (int j = 0; j < n / 2; ++j) {
        sum += w[j] * cosine[at];
        at += 2 * k;
        if (at >= 4 * n) at -= 4 * n;
      }
      c[(size_t)k * F] = sum * (k ? 2.0L : 1.0L) / n;
    }
  });
  for (int q = 0; q < np; ++q) {
    const int p = pairs[q];
    ld gmax = 0.0L;
    for (size_t k = 0; k < (size_t)n * F; ++k)
      gmax = std::max(gmax, std::fabs(val[(size_t)q * n * F + k]));
    terms[p] = 0;
    ld tail = 0.0L;
    for (int k = n - 1; k >= 16; --k) {
      ld a = 0.0L;
      for (int f = 0; f < F; ++f) a = std::max(a, std::fabs(coef[p][(size_t)k * F + f]));
      tail += a;
      if (tail > gmax * 0x1p-55L) break;
      if (k % 16 == 0 && k <= std::min(n - 16, kExpandMaxTerms)) terms[p] = k;
    }
  }
}

}  // namespace

bool build_expansion(const ModelHost& m, ExpandHost& e) {
  const int np = m.ntypes * m.ntypes, F = m.emb[2];
  // (finite parameters give finite coefficients: every layer is a tanh)
  for (const auto* v : {&m.emb_params, &m.davg, &m.dstd})
    for (double x : *v)
      if (!std::isfinite(x)) return false;
  std::vector<std::vector<ld>> coef(np);
  std::vector<int> terms(np, 0);
  for (const int n : {112, 176, 304}) {
    std::vector<int> todo;
    for (int p = 0; p < np; ++p)
      if (terms[p] == 0) todo.push_back(p);
    if (!todo.empty()) coefficients(m, todo, n, coef, terms);
  }
  if (*std::min_element(terms.begin(), terms.end()) == 0) return false;
  const int most = *std::max_element(terms.begin(), terms.end());
  e.H = most <= 64 ? 1 : most <= 128 ? 2 : 4;
  const int N = 64 * e.H, NU2 = expand_nu2(F), NQ2 = expand_nq2(F);
  const long fs = expand_fwd_stride(e.H, F), bs = expand_bwd_stride(e.H, F);
  e.fwd.assign((size_t)np * fs, 0.0);
  e.bwd.assign((size_t)np * bs, 0.0);
  e.blocks.assign(np, 0);
  for (int p = 0; p < np; ++p) {
    e.blocks[p] = terms[p] / 16;
    std::vector<ld> c((size_t)N * F, 0.0L);
    std::copy_n(coef[p].begin(), (size_t)terms[p] * F, c.begin());
    to_products(c.data(), N, 64, F);
    for (int h = 0; h < N; h += 64) to_products(c.data() + (size_t)h * F, 64, 16, F);
    for (int h = 0; h < N; h += 16) to_products(c.data() + (size_t)h * F, 16, 4, F);
    // (a product expansion of a polynomial of degree < 16 blocks has no terms
    // beyond those blocks: each conversion only moves weight downwards)
    for (int k = 0; k < N; ++k)
      for (int f = 0; f < F; ++f) {
        const double v = (double)c[(size_t)k * F + f];
        const int u = f / 16;
        e.fwd[p * fs + (((long)(k / 4) * NU2 + u / 2) * 64 + 16 * (k % 4) + f % 16) * 2 + u % 2] = v;
        e.bwd[p * bs + (((long)(k / 16) * NQ2 + f / 8) * 64 + 16 * (f % 8 / 2) + k % 16) * 2 +
              f % 2] = v;
      }
  }
  // basis values of a padded slot (y = 0)
  const ld x = -(ld)kExpandB;
  auto cheb = [&](int n) { return std::cos(n * std::acos(x)); };
  e.phi_pad.resize(N);
  for (int k = 0; k < N; ++k)
    e.phi_pad[k] = (double)(cheb(k / 64 * 64) * cheb(k / 16 % 4 * 16) * cheb(k / 4 % 4 * 4) * cheb(k % 4));
  return true;
}

}  // namespace dpamd
