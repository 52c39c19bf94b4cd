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

// tanh by the addition formula: a = k / 32 nearest to |x| from a table, the rest
// b (|b| <= 1/64) from its series, truncated below 2^-66 of b. The C library's
// takes 80 ns, most of a net's evaluation; this 15.
ld tanh_ld(ld x) {
  constexpr int N = 24 * 32;  // 1 - tanh(24) < 2^-66
  static const std::vector<ld> table = [] {
    std::vector<ld> t(N + 1);
    for (int k = 0; k <= N; ++k) t[k] = std::tanh((ld)k / 32);
    return t;
  }();
  const ld v = std::fabs(x);
  if (!(v < 24)) return x > 0 ? 1 : -1;
  const int k = (int)(v * 32 + 0.5L);
  const ld b = v - (ld)k / 32, q = b * b, t = table[k];
  constexpr ld c3 = -1.0L / 3, c5 = 2.0L / 15, c7 = -17.0L / 315, c9 = 62.0L / 2835, c11 = -1382.0L / 155925;
  const ld u = b + b * q * (c3 + q * (c5 + q * (c7 + q * (c9 + q * c11))));
  const ld y = (t + u) / (1 + t * u);
  return x < 0 ? -y : y;
}

// z[0 .. C) += x W for C neighbouring columns of a layer: one load of x[q] (an
// extended-precision value in memory costs several cycles) serves C products,
// whose sums stay in registers.
template <int C>
void columns(const ld* x, int in, const double* W, int out, ld* z) {
  ld a[C];
  for (int c = 0; c < C; ++c) a[c] = z[c];
  for (int q = 0; q < in; ++q) {
    const ld v = x[q];
    for (int c = 0; c < C; ++c) a[c] += v * W[(long)q * out + c];
  }
  for (int c = 0; c < C; ++c) z[c] = a[c];
}

// One net at s, in extended precision (x, y: scratch of at least L3 values).
void net_ld(const ModelHost& m, const double* P, ld s, std::vector<ld>& x, std::vector<ld>& y) {
  const int L[4] = {1, m.emb[0], m.emb[1], m.emb[2]};
  x[0] = s;
  for (int k = 0; k < 3; ++k) {
    const int in = L[k], out = L[k + 1];
    const double* W = P;
    const double* b = P + (long)in * out;
    P = b + out;
    std::copy_n(b, out, y.begin());
    int f = 0;
    for (; f + 4 <= out; f += 4) columns<4>(x.data(), in, W + f, out, y.data() + f);
    for (; f < out; ++f) columns<1>(x.data(), in, W + f, out, y.data() + f);
    for (f = 0; f < out; ++f)
      y[f] = tanh_ld(y[f]) + (out == in && k > 0 ? x[f] : out == 2 * in && k > 0 ? x[f % in] : 0.0L);
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
// enough that the derivative's truncation stays below its rounding too. The
// last 16 coefficients come first: where they alone are larger than that (excess,
// their sum in units of it, above 1), no number of terms will do, and the others
// are not formed.
void coefficients(const ModelHost& m, const std::vector<int>& pairs, int n,
                  std::vector<std::vector<ld>>& coef, std::vector<int>& terms,
                  std::vector<ld>& excess) {
  constexpr int C = 4;  // features formed together (L3 is a multiple)
  const int np = (int)pairs.size(), F = m.emb[2], NF = F / C;
  const ld pi = 3.14159265358979323846264338327950288L;
  std::vector<ld> cosine(4 * n);  // cos(i pi / 2n): exact angles for cos(k (2j + 1) pi / 2n)
  for (int i = 0; i < 4 * n; ++i) cosine[i] = std::cos((ld)i * pi / (2 * n));
  std::vector<ld> val((size_t)np * n * F);  // [pair][node][feature]
  parallel(np * n, [&](int k) {
    const int p = pairs[k / n], j = k % n;
    const ld z = (cosine[2 * j + 1] + (ld)kExpandB) / (ld)kExpandA;
    const ld s = (z / (2 - z) / (ld)kExpandRmin - (ld)m.davg[(size_t)p * 4]) / (ld)m.dstd[(size_t)p * 4];
    std::vector<ld> x(F), y(F);
    net_ld(m, m.emb_params.data() + (size_t)p * m.emb_block, s, x, y);
    std::copy_n(x.begin(), F, val.begin() + (size_t)k * F);
  });
  for (int p : pairs) coef[p].assign((size_t)n * F, 0.0L);
  // coefficients k0 .. k1 - 1 of features C q .. C q + C - 1 of pair pairs[i]
  auto transform = [&](int i, int q, int k0, int k1) {
    const ld* v = val.data() + (size_t)i * n * F + C * q;
    ld* c = coef[pairs[i]].data() + C * q;
    // node n - 1 - j lies opposite node j: T_k there is (-1)^k T_k here
    std::vector<ld> fold((size_t)n * C);
    for (int j = 0; j < n / 2; ++j)
      for (int f = 0; f < C; ++f) {
        const ld a = v[(size_t)j * F + f], b = v[(size_t)(n - 1 - j) * F + f];
        fold[j * C + f] = a + b;
        fold[(n / 2 + j) * C + f] = a - b;
      }
    for (int k = k0; k < k1; ++k) {
      const ld* w = fold.data() + (k % 2 ? n / 2 * C : 0);
      ld sum[C] = {};
      int at = k;  // k (2j + 1) mod 4n
      for (int j = 0; j < n / 2; ++j) {
        const ld t = cosine[at];
        for (int f = 0; f < C; ++f) sum[f] += t * w[j * C + f];
        at += 2 * k;
        if (at >= 4 * n) at -= 4 * n;
      }
      for (int f = 0; f < C; ++f) c[(size_t)k * F + f] = sum[f] * (k ? 2.0L : 1.0L) / n;
    }
  };
  // sum over k0 <= k < k1 of the largest |coefficient| of a feature
  auto tail = [&](int i, int k0, int k1) {
    ld sum = 0.0L;
    for (int k = k0; k < k1; ++k) {
      ld a = 0.0L;
      for (int f = 0; f < F; ++f) a = std::max(a, std::fabs(coef[pairs[i]][(size_t)k * F + f]));
      sum += a;
    }
    return sum;
  };
  parallel(np * NF, [&](int q) { transform(q / NF, q % NF, n - 16, n); });
  std::vector<ld> limit(np, 0.0L), last(np);
  parallel(np, [&](int i) {
    for (size_t k = 0; k < (size_t)n * F; ++k)
      limit[i] = std::max(limit[i], std::fabs(val[(size_t)i * n * F + k]));
    limit[i] *= 0x1p-55L;
    last[i] = tail(i, n - 16, n);
  });
  std::vector<int> good;  // positions in pairs
  for (int i = 0; i < np; ++i) {
    terms[pairs[i]] = 0;
    if (last[i] <= limit[i]) good.push_back(i);
    else excess[pairs[i]] = limit[i] > 0 ? last[i] / limit[i] : last[i];
  }
  parallel((int)good.size() * NF, [&](int q) { transform(good[q / NF], q % NF, 0, n - 16); });
  for (int i : good) {
    ld sum = last[i];
    for (int k = n - 16; k >= 16 && sum <= limit[i]; k -= 16) {
      if (k <= kExpandMaxTerms) terms[pairs[i]] = k;
      sum += tail(i, k - 16, k);
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
  std::vector<ld> excess(np, 0.0L);
  std::vector<int> todo(np);
  for (int p = 0; p < np; ++p) todo[p] = p;
  auto expand = [&](const std::vector<int>& pairs, int n) {
    coefficients(m, pairs, n, coef, terms, excess);
    todo.clear();
    for (int p = 0; p < np; ++p)
      if (terms[p] == 0) todo.push_back(p);
  };
  expand(todo, 112);
  if (!todo.empty()) {
    // the steepest net decides alone whether there is an expansion for all:
    // a model that has none costs little more than the first attempt
    const int worst = *std::max_element(todo.begin(), todo.end(),
                                        [&](int p, int q) { return excess[p] < excess[q]; });
    expand({worst}, 304);
    if (terms[worst] == 0) return false;
  }
  for (const int n : {176, 304})
    if (!todo.empty()) expand(std::vector<int>(todo), n);
  if (!todo.empty()) return false;
  const int most = *std::max_element(terms.begin(), terms.end());
  e.H = most <= 64 ? 1 : most <= 128 ? 2 : 4;
  const int N = 64 * e.H, NU2 = expand_nu2(F), NQ2 = expand_nq2(F);
  const long fs = expand_fwd_stride(e.H, F), bs = expand_bwd_stride(e.H, F);
  e.fwd.assign((size_t)np * fs, 0.0);
  e.bwd.assign((size_t)np * bs, 0.0);
  e.blocks.assign(np, 0);
  parallel(np, [&](int p) {
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
  });
  // basis values of a padded slot (y = 0)
  const ld x = -(ld)kExpandB;
  auto cheb = [&](int n) { return std::cos(n * std::acos(x)); };
  e.phi_pad.resize(N);
  for (int k = 0; k < N; ++k)
    e.phi_pad[k] = (double)(cheb(k / 64 * 64) * cheb(k / 16 % 4 * 16) * cheb(k / 4 % 4 * 4) * cheb(k % 4));
  return true;
}

}  // namespace dpamd
