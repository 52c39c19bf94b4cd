// Host side of the embedding nets' expansion (expand.h): coefficients by
// Chebyshev interpolation in extended precision, their check, and the layouts
// the kernels read.
#include "expand.h"

#include <pthread.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <exception>
#include <mutex>
#include <type_traits>

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

// One net at s, in extended precision: features [L3].
constexpr int kWidest = 128;
void net_ld(const ModelHost& m, const double* P, ld s, ld* features) {
  const int L[4] = {1, m.emb[0], m.emb[1], m.emb[2]};
  ld buf[2][kWidest], *x = buf[0], *y = buf[1];
  x[0] = s;
  for (int k = 0; k < 3; ++k) {
    const int in = L[k], out = L[k + 1];
    const double* W = P;
    const double* b = P + (long)in * out;
    P = b + out;
    std::copy_n(b, out, y);
    int f = 0;
    for (; f + 4 <= out; f += 4) columns<4>(x, in, W + f, out, y + f);
    for (; f < out; ++f) columns<1>(x, in, W + f, out, y + f);
    for (f = 0; f < out; ++f)
      y[f] = tanh_ld(y[f]) + (out == in && k > 0 ? x[f] : out == 2 * in && k > 0 ? x[f % in] : 0.0L);
    std::swap(x, y);
  }
  std::copy_n(x, L[3], features);
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

// The host threads of one build (up to 8 with the caller's), started once: a
// start costs as much as a phase of a small model. Their stacks are small, so
// that the C library keeps them for the next build: stacks of the default 8 MB
// are mostly unmapped, and the device allocations of the handle's first
// evaluation then land at addresses the card has no page tables for yet (1.3
// against 0.5 ms for 864 Cu atoms where a handle replaces another).
class Team {
 public:
  Team() {
    pthread_attr_t attr;
    if (pthread_attr_init(&attr) != 0) return;
    (void)pthread_attr_setstacksize(&attr, 256 * 1024);
    // (if fewer threads than asked for: their work stays with the caller)
    while (size_ < kThreads && pthread_create(&pool_[size_], &attr, serve, this) == 0) ++size_;
    (void)pthread_attr_destroy(&attr);
  }
  ~Team() {
    {
      std::lock_guard<std::mutex> lock(m_);
      stop_ = true;
    }
    wake_.notify_all();
    for (size_t q = 0; q < size_; ++q) pthread_join(pool_[q], nullptr);
  }
  Team(const Team&) = delete;
  Team& operator=(const Team&) = delete;

  // f(0) .. f(n - 1), in any order. What an f throws ends the others' work too
  // and is thrown again once every thread has stopped.
  template <class Fn>
  void run(int n, Fn&& f) {
    {
      std::lock_guard<std::mutex> lock(m_);
      call_ = [](void* g, int k) { (*static_cast<std::remove_reference_t<Fn>*>(g))(k); };
      f_ = &f;
      n_ = n;
      next_ = 0;
      failed_ = false;
      error_ = nullptr;
      busy_ = size_;
      ++round_;
    }
    wake_.notify_all();
    work();
    std::unique_lock<std::mutex> lock(m_);
    done_.wait(lock, [this]() { return busy_ == 0; });
    if (error_) std::rethrow_exception(error_);
  }

 private:
  void work() {
    try {
      for (int k = next_++; k < n_ && !failed_; k = next_++) call_(f_, k);
    } catch (...) {
      if (!failed_.exchange(true)) error_ = std::current_exception();
    }
  }
  static void* serve(void* self) {
    Team& t = *static_cast<Team*>(self);
    long seen = 0;
    std::unique_lock<std::mutex> lock(t.m_);
    for (;;) {
      t.wake_.wait(lock, [&]() { return t.stop_ || t.round_ != seen; });
      if (t.stop_) return nullptr;
      seen = t.round_;
      lock.unlock();
      t.work();
      lock.lock();
      if (--t.busy_ == 0) t.done_.notify_one();
    }
  }

  static constexpr size_t kThreads = 7;
  std::mutex m_;
  std::condition_variable wake_, done_;
  pthread_t pool_[kThreads];
  size_t size_ = 0;
  // the phase: set by run() under the lock, before the threads are woken
  void (*call_)(void*, int) = nullptr;
  void* f_ = nullptr;
  int n_ = 0;
  std::atomic<int> next_{0};
  std::atomic<bool> failed_{false};
  std::exception_ptr error_;  // written by the thread that sets failed_
  size_t busy_ = 0;           // threads that have not finished the phase
  long round_ = 0;
  bool stop_ = false;
};

// Chebyshev coefficients [n][L3] of the nets of `pairs` from n nodes (even),
// and per pair the number of terms (a multiple of 16, 0 if none will do) past
// which the magnitudes of every feature's coefficients sum to at most 2^-55
// of the largest feature: below the rounding of the sum itself, and small
// enough that the derivative's truncation stays below its rounding too. The
// last 16 coefficients come first: where they alone are larger than that (excess,
// their sum in units of it, above 1), no number of terms will do, and the others
// are not formed.
constexpr int kMostNodes = 304;
void coefficients(Team& team, const ModelHost& m, const std::vector<int>& pairs, int n,
                  std::vector<std::vector<ld>>& coef, std::vector<int>& terms,
                  std::vector<ld>& excess) {
  constexpr int C = 4;  // features formed together (L3 is a multiple)
  const int np = (int)pairs.size(), F = m.emb[2], NF = F / C;
  const ld pi = 3.14159265358979323846264338327950288L;
  std::vector<ld> cosine(4 * n);  // cos(i pi / 2n): exact angles for cos(k (2j + 1) pi / 2n)
  for (int i = 0; i < 4 * n; ++i) cosine[i] = std::cos((ld)i * pi / (2 * n));
  std::vector<ld> val((size_t)np * n * F);  // [pair][node][feature]
  for (int p : pairs) coef[p].assign((size_t)n * F, 0.0L);
  team.run(np * n, [&](int k) {
    const int p = pairs[k / n], j = k % n;
    const ld z = (cosine[2 * j + 1] + (ld)kExpandB) / (ld)kExpandA;
    const ld s = (z / (2 - z) / (ld)kExpandRmin - (ld)m.davg[(size_t)p * 4]) / (ld)m.dstd[(size_t)p * 4];
    net_ld(m, m.emb_params.data() + (size_t)p * m.emb_block, s, val.data() + (size_t)k * F);
  });
  // coefficients k0 .. k1 - 1 of features C q .. C q + C - 1 of pair pairs[i]
  auto transform = [&](int i, int q, int k0, int k1) {
    const ld* v = val.data() + (size_t)i * n * F + C * q;
    ld* c = coef[pairs[i]].data() + C * q;
    // node n - 1 - j lies opposite node j: T_k there is (-1)^k T_k here
    ld fold[kMostNodes * C];
    for (int j = 0; j < n / 2; ++j)
      for (int f = 0; f < C; ++f) {
        const ld a = v[(size_t)j * F + f], b = v[(size_t)(n - 1 - j) * F + f];
        fold[j * C + f] = a + b;
        fold[(n / 2 + j) * C + f] = a - b;
      }
    for (int k = k0; k < k1; ++k) {
      const ld* w = fold + (k % 2 ? n / 2 * C : 0);
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
  team.run(np * NF, [&](int q) { transform(q / NF, q % NF, n - 16, n); });
  std::vector<ld> limit(np, 0.0L), last(np);
  team.run(np, [&](int i) {
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
  team.run((int)good.size() * NF, [&](int q) { transform(good[q / NF], q % NF, 0, n - 16); });
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
  Team team;
  std::vector<ld> excess(np, 0.0L);
  std::vector<int> todo(np);
  for (int p = 0; p < np; ++p) todo[p] = p;
  auto expand = [&](const std::vector<int>& pairs, int n) {
    coefficients(team, m, pairs, n, coef, terms, excess);
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
    expand({worst}, kMostNodes);
    if (terms[worst] == 0) return false;
  }
  for (const int n : {176, kMostNodes})
    if (!todo.empty()) expand(std::vector<int>(todo), n);
  if (!todo.empty()) return false;
  const int most = *std::max_element(terms.begin(), terms.end());
  e.H = most <= 64 ? 1 : most <= 128 ? 2 : 4;
  const int N = 64 * e.H, NU2 = expand_nu2(F), NQ2 = expand_nq2(F);
  const long fs = expand_fwd_stride(e.H, F), bs = expand_bwd_stride(e.H, F);
  e.fwd.assign((size_t)np * fs, 0.0);
  e.bwd.assign((size_t)np * bs, 0.0);
  e.blocks.assign(np, 0);
  std::vector<ld> prod((size_t)np * N * F, 0.0L);
  team.run(np, [&](int p) {
    e.blocks[p] = terms[p] / 16;
    ld* c = prod.data() + (size_t)p * N * F;
    std::copy_n(coef[p].begin(), (size_t)terms[p] * F, c);
    to_products(c, N, 64, F);
    for (int h = 0; h < N; h += 64) to_products(c + (size_t)h * F, 64, 16, F);
    for (int h = 0; h < N; h += 16) to_products(c + (size_t)h * F, 16, 4, F);
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
