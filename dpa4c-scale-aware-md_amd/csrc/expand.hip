// Environment matrix + embedding + descriptor contraction, and its backward,
// with the embedding nets expanded in one variable per slot (expand.h), on
// gfx950 FP64 MFMA (v_mfma_f64_16x16x4f64). Both precision modes use these
// kernels (fp64 throughout; E is the element type of T and dE/dT in memory),
// unless some net of the model has no short enough expansion; embed.hip and
// embed_f32.hip then evaluate the nets slot by slot.
//
// Work unit: one wave (W = 1: a block of its own, nothing is shared, so there
// is no barrier and no tail) owns four consecutive centres of one type; lane
// group g (lane = 16 g + c) walks the slots of centre g, 16 at a time. Systems
// with too few centres to fill the device give the four centres to a block of
// W = 4 waves that share out the rounds and the products' tiles. A round prepares 64 slots, one a lane (environment row, basis
// values), in LDS; the products then read them per centre.
//
// Forward, per neighbour section: M[(m, b)][(p, l)] += R[m] T_16b (x) T_4p T_l
// over the slots, four slots (k) per MFMA: 16 rows (m, b), 16 columns (p, l),
// one accumulator per group of 64 terms and centre. At the section's end the
// four centres' M ([16 rows = (m, centre)][terms], through LDS) is multiplied
// by the section's coefficients into T [16][L3], which is kept over the
// sections and written once. The section's padded slots enter as one slot of
// weight npad in M's initial value.
//
// Backward, per section: dM [16 rows][terms] = dE/dT C^T, rearranged through
// LDS into the A operands [(m, b)][(p, l)] of each centre; then per tile of
// 16 slots of a centre Y = dM (T_4p T_l) and Y' = dM (T_4p T_l)' (4 k-steps
// each), so that lane (g = b, c = slot) holds Y[m] for m = 0..3, and
//   u[m] = sum_b T_16b Y[m],  v = sum_b sum_m R[m] (T_16b Y[m])'
// are summed over the lane groups. The edge gradient and its outputs are
// formed with one slot a lane again; each lane's own sums belong to one
// centre over all rounds and sections.
//
// What bounds them: fp64 issue, MFMA and VALU together (they never overlap
// for fp64 on gfx950). Per centre of 138 slots and 80 terms the forward
// issues 70 MFMAs for M and 40 for T against 15,500 for the nets.
//
// Reference analogs: the tabulated radial + PairFiLM embedding
// include/dpa_chain/graph_compress.cuh:91-154 and the per-row moment
// accumulation deepmd-op/overlays/op/pt/dpa4c/raw_kernel.cuh:71-120.
#include "env.h"
#include "expand.h"
#include "kernels.h"

namespace dpamd {

namespace {

template <class E>
struct alignas(2 * sizeof(E)) Vec2 {
  E x, y;
};

// Environment row of a slot (as env_value) and the expansion's y.
__device__ __forceinline__ double env_row(const ExpandArgs& a, double d0, double d1, double d2,
                                          const double* avg, const double* isd, double* Rn) {
  const double r2 = d0 * d0 + d1 * d1 + d2 * d2;
  const double inv_r = inv_sqrt(r2);
  double dsw;
  const double sw = switch5(r2 * inv_r, a.rcut_smth, a.rcut, a.inv_sw, &dsw);
  const double sr = sw * inv_r, q = sr * inv_r;
  Rn[0] = (sr - avg[0]) * isd[0];
  Rn[1] = (q * d0 - avg[1]) * isd[1];
  Rn[2] = (q * d1 - avg[2]) * isd[2];
  Rn[3] = (q * d2 - avg[3]) * isd[3];
  return kExpandRmin * sr;
}

// 1 / (1 + y), y >= 0
__device__ __forceinline__ double inv_1p(double y) {
  const double w = 1.0 + y;
  double v = __builtin_amdgcn_rcp(w);
  v = fma(fma(-w, v, 1.0), v, v);
  return fma(fma(-w, v, 1.0), v, v);
}

// LDS written by the block's waves made visible to them (W = 1: to the wave)
template <int W>
__device__ __forceinline__ void block_sync() {
  if constexpr (W > 1) __syncthreads();
  else wave_lds_sync();
}

// sum over the 16 lanes of a lane group, in every lane
__device__ __forceinline__ double sum_c16(double v) {
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o, kWave);
  return v;
}

__device__ __forceinline__ int lane_int(int v, int lane) {
  return __builtin_amdgcn_readlane(v, lane);
}
__device__ __forceinline__ double lane_double(double v, int lane) {
  return from32(__builtin_amdgcn_readlane(hi32(v), lane), __builtin_amdgcn_readlane(lo32(v), lane));
}

// One net at s, evaluated by the whole wave (slots closer than kExpandRmin,
// outside the expansion's range): G and, with TAN, dG/ds of features lane and
// lane + 64. net = W1 b1 W2 b2 W3 b3 as in the model file; x: LDS scratch of
// 2 (L1 + L2) doubles.
template <bool TAN>
__device__ __forceinline__ void net_at(const double* net, const int* L, double s, double* x,
                                       int lane, double G[2], double dG[2]) {
  const int L1 = L[0], L2 = L[1], L3 = L[2];
  double *x1 = x, *t1 = x + L1, *x2 = x + 2 * L1, *t2 = x2 + L2;
  const double* W2 = net + 2 * L1;
  const double* W3 = W2 + L1 * L2 + L2;
  wave_lds_sync();
  if (lane < L1) {
    const double w = net[lane], y = tanh(fma(s, w, net[L1 + lane]));
    x1[lane] = y;
    t1[lane] = (1.0 - y * y) * w;
  }
  wave_lds_sync();
  if (lane < L2) {
    double z = 0.0, zt = 0.0;
    for (int k = 0; k < L1; ++k) {
      const double w = W2[k * L2 + lane];
      z = fma(x1[k], w, z);
      if constexpr (TAN) zt = fma(t1[k], w, zt);
    }
    const double y = tanh(z + W2[L1 * L2 + lane]);
    const int q = lane % L1;
    const bool res = L2 == L1 || L2 == 2 * L1;
    x2[lane] = y + (res ? x1[q] : 0.0);
    t2[lane] = (1.0 - y * y) * zt + (res ? t1[q] : 0.0);
  }
  wave_lds_sync();
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int f = lane + 64 * e;
    G[e] = 0.0;
    dG[e] = 0.0;
    if (f < L3) {
      double z = 0.0, zt = 0.0;
      for (int k = 0; k < L2; ++k) {
        const double w = W3[k * L3 + f];
        z = fma(x2[k], w, z);
        if constexpr (TAN) zt = fma(t2[k], w, zt);
      }
      const double y = tanh(z + W3[L2 * L3 + f]);
      const int q = f % L2;
      const bool res = L3 == L2 || L3 == 2 * L2;
      G[e] = y + (res ? x2[q] : 0.0);
      if constexpr (TAN) dG[e] = (1.0 - y * y) * zt + (res ? t2[q] : 0.0);
    }
  }
}

// Consecutive waves (neighbouring centres) on one XCD: the hardware deals
// blocks to the XCDs round robin. A bijection on the grid.
__device__ __forceinline__ int xcd_wave() {
  const int nb = gridDim.x, q = nb / kXcds, r = nb % kXcds, x = blockIdx.x % kXcds;
  return x * q + (x < r ? x : r) + (int)blockIdx.x / kXcds;
}

// The wave's four centres: type, first bucket position, this lane group's.
struct Centres {
  int ti, pos0, i;
  bool ok;
};
__device__ __forceinline__ Centres my_centres(const ExpandArgs& a, int g) {
  const int w = xcd_wave();
  Centres q;
  q.ti = 0;
  while (q.ti + 1 < a.ntypes && w >= a.wave_off[q.ti + 1]) ++q.ti;
  q.pos0 = a.type_off[q.ti] + 4 * (w - a.wave_off[q.ti]);
  const int last = a.type_off[q.ti + 1] - 1;
  q.ok = q.pos0 + g <= last;
  q.i = a.items[min(q.pos0 + g, last)];
  return q;
}

constexpr int kRecF(int H) { return H > 2 ? 17 : 15; }  // odd: lanes' rows in distinct banks
constexpr int kRecB(int H) { return H > 2 ? 30 : 26; }  // 16-byte reads: distinct banks
constexpr int kTr = 68;  // row stride of the 64-term transposition buffer (4 mod 32)

constexpr int fwd_lds(int H) {
  const int rec = 64 * kRecF(H), m = 16 * (64 * H + 4);
  return rec > m ? rec : m;
}
constexpr int bwd_lds(int H) { return 64 * kRecB(H); }
static_assert(bwd_lds(1) >= 16 * kTr, "transposition buffer fits a wave's records");
static_assert(fwd_lds(1) >= 2 * (32 + 64) && bwd_lds(1) >= 2 * (32 + 64), "net_at scratch");

}  // namespace

template <class E, int NU3, int H, int W>
__global__ __launch_bounds__(64 * W, H > 2 ? 1 : 2) void k_expand_fwd(ExpandArgs a) {
  extern __shared__ __align__(16) double lds_all[];
  constexpr int RS = kRecF(H), LD = 64 * H + 4, NU2 = (NU3 + 1) / 2;
  constexpr int NT = (NU3 + W - 1) / W;  // T tiles of a wave: u = W k + w
  const int w = W > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  double* lds = lds_all + w * fwd_lds(H);
  const Centres q4 = my_centres(a, g);
  const int ti = q4.ti, L3 = a.emb[2];
  const double xi = a.ext[3L * q4.i], yi = a.ext[3L * q4.i + 1], zi = a.ext[3L * q4.i + 2];
  // this lane's record entries: T_l, T_4p (column c = 4p + l) and T_16b, R[m]
  // (row c = 4m + b)
  const int eL = c & 3, eP = (c >> 2) ? 3 + (c >> 2) : 0, eB = (c & 3) ? 6 + (c & 3) : 0;
  const int eR = 10 + (c >> 2);
  double* rec = lds + lane * RS;
  d4 T[NT];
#pragma unroll
  for (int u = 0; u < NT; ++u) T[u] = d4{0.0, 0.0, 0.0, 0.0};
  bool close = false;  // some slot of this lane is outside the expansion

  for (int tj = 0; tj < a.ntypes; ++tj) {
    const int pair = ti * a.ntypes + tj, nblk = a.blocks[pair];
    double avg[4], isd[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      avg[m] = a.envp[pair * 8 + m];
      isd[m] = 1.0 / a.envp[pair * 8 + 4 + m];
    }
    const int nr = q4.ok ? a.nreal[(long)q4.i * a.ntypes + tj] : 0;
    const int* row = a.nlist + (long)q4.i * a.nnei + a.sec[tj];
    const int slast = a.sel[tj] - 1;
    int nrj[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) nrj[j] = lane_int(nr, 16 * j);
    const int most = max(max(nrj[0], nrj[1]), max(nrj[2], nrj[3]));
    // the padded slots: R = -avg / std at y = 0 (absent centres: any value,
    // they are not written)
    d4 acc[4][H];
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const double pp = a.phi_pad[64 * h + lane];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const double np = w == 0 ? (double)(a.sel[tj] - nrj[j]) * pp : 0.0;
#pragma unroll
        for (int m = 0; m < 4; ++m) acc[j][h][m] = np * (-avg[m] * isd[m]);
      }
    }
    // coordinates one round ahead, indices two (clamped into the section)
    double nx = 0.0, ny = 0.0, nz = 0.0;
    const int s0 = 16 * w + c;
    if (s0 < nr) {
      const long j = row[s0];
      nx = a.ext[3 * j];
      ny = a.ext[3 * j + 1];
      nz = a.ext[3 * j + 2];
    }
    int jn = row[min(s0 + 16 * W, slast)];
    for (int t = 16 * w; t < most; t += 16 * W) {
      const int slot = t + c;
      double Rn[4] = {0.0, 0.0, 0.0, 0.0}, x = 0.0;
      if (slot < nr) {
        const double y = env_row(a, nx - xi, ny - yi, nz - zi, avg, isd, Rn);
        x = fma(kExpandA * 2.0 * y, inv_1p(y), -kExpandB);
        if (y > 1.0) {
          close = true;
          x = 0.0;
          Rn[0] = Rn[1] = Rn[2] = Rn[3] = 0.0;
        }
      }
      if (slot + 16 * W < nr) {
        nx = a.ext[3L * jn];
        ny = a.ext[3L * jn + 1];
        nz = a.ext[3L * jn + 2];
      }
      jn = row[min(slot + 32 * W, slast)];
      double v[kNumBasis<H>];
      basis_values<H>(x, v);
      wave_lds_sync();
#pragma unroll
      for (int k = 0; k < 10; ++k) rec[k] = v[k];
#pragma unroll
      for (int m = 0; m < 4; ++m) rec[10 + m] = Rn[m];
#pragma unroll
      for (int h = 1; h < H; ++h) rec[13 + h] = v[9 + h];
      wave_lds_sync();
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (t >= nrj[j]) continue;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double* r = lds + (16 * j + 4 * q + g) * RS;
          const double chi = r[eL] * r[eP], av = r[eB] * r[eR];
          acc[j][0] = mfma_f64(av, chi, acc[j][0]);
#pragma unroll
          for (int h = 1; h < H; ++h) acc[j][h] = mfma_f64(av * r[13 + h], chi, acc[j][h]);
        }
      }
    }
    // T += M C: row 4m + j of M in LDS is A's row
    wave_lds_sync();
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int h = 0; h < H; ++h)
#pragma unroll
        for (int m = 0; m < 4; ++m) lds[(4 * m + j) * LD + 64 * h + lane] = acc[j][h][m];
    const int nq = 4 * nblk;
    if constexpr (W == 1) {
      wave_lds_sync();
      const double2* C = reinterpret_cast<const double2*>(a.cf) + (long)pair * (a.cf_stride / 2) + lane;
      const double* A = lds + c * LD + g;
      double2 b0[NU2], b1[NU2];
#pragma unroll
      for (int u = 0; u < NU2; ++u) {
        b0[u] = C[64 * u];
        b1[u] = C[64 * (NU2 + u)];
      }
      for (int q = 0; q < nq; q += 2) {
        const double a0 = A[4 * q], a1 = A[4 * q + 4];
        const double2* Cn = C + 64L * NU2 * min(q + 2, nq - 2);
#pragma unroll
        for (int u = 0; u < NU3; ++u) T[u] = mfma_f64(a0, u & 1 ? b0[u / 2].y : b0[u / 2].x, T[u]);
#pragma unroll
        for (int u = 0; u < NU2; ++u) b0[u] = Cn[64 * u];
#pragma unroll
        for (int u = 0; u < NU3; ++u) T[u] = mfma_f64(a1, u & 1 ? b1[u / 2].y : b1[u / 2].x, T[u]);
#pragma unroll
        for (int u = 0; u < NU2; ++u) b1[u] = Cn[64 * (NU2 + u)];
      }
    } else {
      // the waves' shares of M are added where they are read; each wave its
      // tiles u = W k + w of T, four k-steps' coefficients in flight
      __syncthreads();
      const double* A = lds_all + c * LD + g;
      const double* C = a.cf + (long)pair * a.cf_stride + 2 * lane;
      for (int q = 0; q < nq; q += 4) {
        double av[4], b[4][NT];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int k = 0; k < NT; ++k) {
            const int u = min(W * k + w, NU3 - 1);
            b[e][k] = C[128L * (NU2 * (q + e) + u / 2) + (u & 1)];
          }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          av[e] = A[4 * (q + e)];
#pragma unroll
          for (int v = 1; v < W; ++v) av[e] += A[v * fwd_lds(H) + 4 * (q + e)];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int k = 0; k < NT; ++k) T[k] = mfma_f64(av[e], b[e][k], T[k]);
      }
      __syncthreads();
    }
  }
  // lane (g, c): T of centre g (bucket position pos0 + g), features 16u + c
  E* Tt = static_cast<E*>(a.Tt) + 4L * (q4.pos0 + g);
  if (q4.ok) {
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const int f = 16 * (W * u + w) + c;
      if (f < L3) {
        Vec4<E> o;
        o.x = (E)(T[u][0] * a.inv_nnei);
        o.y = (E)(T[u][1] * a.inv_nnei);
        o.z = (E)(T[u][2] * a.inv_nnei);
        o.w = (E)(T[u][3] * a.inv_nnei);
        *reinterpret_cast<Vec4<E>*>(Tt + f * a.ldt) = o;
      }
    }
  }
  // slots outside the expansion's range (rare): the net itself, added to the
  // centre's T, which this block alone writes
  bool any = __ballot(close) != 0;
  if constexpr (W > 1) any = __syncthreads_or(any);
  if (__builtin_expect(any, 0)) {
    __threadfence();
    if constexpr (W > 1) __syncthreads();
  }
  if (__builtin_expect(any && w == 0, 0)) {
    for (int j = 0; j < 4; ++j) {
      const int i = lane_int(q4.i, 16 * j);
      const double x0 = lane_double(xi, 16 * j), y0 = lane_double(yi, 16 * j),
                   z0 = lane_double(zi, 16 * j);
      if (!lane_int(q4.ok, 16 * j)) continue;
      for (int tj = 0; tj < a.ntypes; ++tj) {
        const int pair = ti * a.ntypes + tj;
        const int nr = a.nreal[(long)i * a.ntypes + tj];
        double avg[4], isd[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          avg[m] = a.envp[pair * 8 + m];
          isd[m] = 1.0 / a.envp[pair * 8 + 4 + m];
        }
        for (int t = 0; t < nr; t += 64) {
          double Rn[4], y = 0.0;
          if (t + lane < nr) {
            const long k = a.nlist[(long)i * a.nnei + a.sec[tj] + t + lane];
            y = env_row(a, a.ext[3 * k] - x0, a.ext[3 * k + 1] - y0, a.ext[3 * k + 2] - z0, avg, isd, Rn);
          }
          for (unsigned long long todo = __ballot(y > 1.0); todo; todo &= todo - 1) {
            const int src = __ffsll((long long)todo) - 1;
            double R[4], G[2], dG[2];
#pragma unroll
            for (int m = 0; m < 4; ++m) R[m] = lane_double(Rn[m], src);
            net_at<false>(a.nets + (long)pair * a.net_stride, a.emb, R[0], lds, lane, G, dG);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const int f = lane + 64 * e;
              if (f >= L3) continue;
              E* o = static_cast<E*>(a.Tt) + f * a.ldt + 4L * (q4.pos0 + j);
#pragma unroll
              for (int m = 0; m < 4; ++m) {
                // (past the L1, which may hold the line from another wave's turn)
                const double old = (double)__hip_atomic_load(o + m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(o + m, (E)(old + R[m] * G[e] * a.inv_nnei), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
              }
            }
          }
        }
      }
    }
  }
  // the backward's fixed-point sums, cleared as the blocks end
  const long n = a.zero_count ? (long)*a.zero_count : a.zero_n;
  const long stride = (long)gridDim.x * (64 * W), q0 = (long)blockIdx.x * (64 * W) + threadIdx.x;
  const long words = (a.vacc ? 16 : 4) * n;
  for (long q = q0; q < words; q += stride) a.facc[q] = 0ull;
}

namespace {
// One slot's centre side, one slot a lane: into the lane's own sums (force,
// frame virial), and the edge gradient itself when kept. The neighbour side,
// -g and with AV the atom virial -g (x) d charged to the neighbour, is parked
// in the slot's LDS record (fixed point; values 0..2, the atom in word 3,
// values 4..12) for scatter_records.
template <bool AV>
__device__ __forceinline__ void slot_out(const ExpandArgs& a, long e, int j, const double d[3],
                                         const double gv[3], double own[12],
                                         unsigned long long* rec) {
  const double gm = fmax(fabs(gv[0]), fmax(fabs(gv[1]), fabs(gv[2])));
  if (!(gm <= a.fix_gmax)) atomicOr(a.status, kStatusFixedRange);
  rec[3] = (unsigned long long)j;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    own[c] += gv[c];
    rec[c] = to_fixed(gv[c]);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const double w = -gv[c] * d[q];
      own[3 + 3 * c + q] += w;
      if constexpr (AV) rec[4 + 3 * c + q] = to_fixed(w);
    }
    if (a.edge_grad) a.edge_grad[3 * e + c] = gv[c];
  }
}

// Adds the parked values of nrec records (stride RB words, first at rec0) to
// their atoms' sums. The lanes of one instruction cover whole records, so the
// values of an edge make one request: on MI355X random 64-bit atomics run at
// 24 G requests a second, 54 M single ones (131,072 Cu atoms) in 2.36 ms,
// as 18 M requests of three in 0.77 ms.
template <bool AV, int RB>
__device__ __forceinline__ void scatter_records(const ExpandArgs& a, const double* rec0, int nrec,
                                                int lane) {
  constexpr int P = AV ? 16 : 4;
  const int q = lane % P;
  for (int k = lane / P; k < nrec; k += 64 / P) {
    const auto* r = reinterpret_cast<const unsigned long long*>(rec0 + k * RB);
    const long j = (long)r[3];
    if (j >= 0 && (q < 3 || (AV && q >= 4 && q < 13))) atomicAdd(a.facc + P * j + q, r[q]);
  }
}
}  // namespace

template <class E, int NU3, int H, bool AV, int W>
__global__ __launch_bounds__(64 * W, H > 2 ? 1 : 2) void k_expand_bwd(ExpandArgs a) {
  extern __shared__ __align__(16) double lds_all[];
  constexpr int RB = kRecB(H);
  constexpr int NQ2 = NU3 == 8 ? 16 : 13;  // expand_nq2(L3)
  const int w = W > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  double* lds = lds_all + w * bwd_lds(H);
  const Centres q4 = my_centres(a, g);
  const int ti = q4.ti, L3 = a.emb[2];
  const double xi = a.ext[3L * q4.i], yi = a.ext[3L * q4.i + 1], zi = a.ext[3L * q4.i + 2];
  // dE/dT row of this lane as A operand rows (row c: m = c / 4, centre c % 4)
  const int irow = __shfl(q4.i, 16 * (c & 3), kWave);
  const E* dTrow = static_cast<const E*>(a.dT) + ((long)irow * 4 + (c >> 2)) * L3 + 2 * g;
  double* rec = lds + lane * RB;
  double own[12];
#pragma unroll
  for (int q = 0; q < 12; ++q) own[q] = 0.0;
  bool close = false;

  for (int tj = 0; tj < a.ntypes; ++tj) {
    const int pair = ti * a.ntypes + tj, nblk = a.blocks[pair];
    const int nr = q4.ok ? a.nreal[(long)q4.i * a.ntypes + tj] : 0;
    const long ebase = (long)q4.i * a.nnei + a.sec[tj];
    const int* row = a.nlist + ebase;
    const int slast = a.sel[tj] - 1;
    int nrj[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) nrj[j] = lane_int(nr, 16 * j);
    const int most = max(max(nrj[0], nrj[1]), max(nrj[2], nrj[3]));
    if (a.edge_grad && q4.ok && w == 0)
      for (int s = nr + c; s <= slast; s += 16)
        for (int q = 0; q < 3; ++q) a.edge_grad[3 * (ebase + s) + q] = 0.0;
    if (most == 0) continue;
    double avg[4], isd[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      avg[m] = a.envp[pair * 8 + m];
      isd[m] = 1.0 / a.envp[pair * 8 + 4 + m];
    }
    // dM = dE/dT C^T (k-step 2q + e: feature 8q + 2g + e), 16 terms at a time
    double dMa[4][H][4];
    {
      double dTa[2 * NQ2];
#pragma unroll
      for (int q = 0; q < NQ2; ++q) {
        // (L3 is even)
        const bool in = 8 * q + 7 < 16 * (NU3 - 1) || 8 * q + 2 * g < L3;
        const Vec2<E> v = in ? *reinterpret_cast<const Vec2<E>*>(dTrow + 8 * q) : Vec2<E>{0, 0};
        dTa[2 * q] = (double)v.x;
        dTa[2 * q + 1] = (double)v.y;
      }
      const double2* C = reinterpret_cast<const double2*>(a.cb) + (long)pair * (a.cb_stride / 2) + lane;
#pragma unroll
      for (int h = 0; h < H; ++h) {
        block_sync<W>();
        // (W = 4: wave w forms term block w)
        for (int b = w; b < 4; b += W) {
          d4 acc = d4{0.0, 0.0, 0.0, 0.0};
          if (4 * h + b < nblk) {
            const double2* Cb = C + 64L * NQ2 * (4 * h + b);
            d4 acc1 = d4{0.0, 0.0, 0.0, 0.0};
            double2 cv[NQ2];
#pragma unroll
            for (int q = 0; q < NQ2; ++q) cv[q] = Cb[64 * q];
#pragma unroll
            for (int q = 0; q < NQ2; ++q) {
              acc = mfma_f64(dTa[2 * q], cv[q].x, acc);
              acc1 = mfma_f64(dTa[2 * q + 1], cv[q].y, acc1);
            }
            acc += acc1;
          }
          // lane (g, c): centre g, term 16b + c, register m
#pragma unroll
          for (int m = 0; m < 4; ++m) lds_all[(4 * g + m) * kTr + 16 * b + c] = acc[m];
        }
        block_sync<W>();
        // A operand of centre j: row c = 4m + b, k = 4q + g
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            dMa[j][h][q] = lds_all[(4 * j + (c >> 2)) * kTr + 16 * (c & 3) + 4 * q + g];
      }
    }
    if constexpr (W > 1) __syncthreads();  // the records overlay the transposition buffer
    double nx = 0.0, ny = 0.0, nz = 0.0;
    const int s0 = 16 * w + c;
    int jc = row[min(s0, slast)];
    if (s0 < nr) {
      nx = a.ext[3L * jc];
      ny = a.ext[3L * jc + 1];
      nz = a.ext[3L * jc + 2];
    }
    int jn = row[min(s0 + 16 * W, slast)];
    for (int t = 16 * w; t < most; t += 16 * W) {
      const int slot = t + c;
      bool live = slot < nr;
      const double d[3] = {nx - xi, ny - yi, nz - zi};
      const int jatom = jc;
      double Rn[4] = {0.0, 0.0, 0.0, 0.0}, x = 0.0, dxds = 0.0;
      if (live) {
        const double y = env_row(a, d[0], d[1], d[2], avg, isd, Rn);
        const double iv = inv_1p(y);
        x = fma(kExpandA * 2.0 * y, iv, -kExpandB);
        dxds = (kExpandA * 2.0 * kExpandRmin) * (iv * iv);  // per unit of sw/r
        if (y > 1.0) {
          close = true;
          live = false;
          x = 0.0;
        }
      }
      jc = jn;
      if (slot + 16 * W < nr) {
        nx = a.ext[3L * jn];
        ny = a.ext[3L * jn + 1];
        nz = a.ext[3L * jn + 2];
      }
      jn = row[min(slot + 32 * W, slast)];
      double v[kNumBasis<H>], s[kNumBasis<H>];
      basis_values<H>(x, v);
      basis_slopes<H>(x, v, s);
      wave_lds_sync();
      // record: (value, slope) of each basis factor, then R
#pragma unroll
      for (int k = 0; k < 10; ++k) *reinterpret_cast<double2*>(rec + 2 * k) = double2{v[k], s[k]};
      *reinterpret_cast<double2*>(rec + 20) = double2{Rn[0], Rn[1]};
      *reinterpret_cast<double2*>(rec + 22) = double2{Rn[2], Rn[3]};
#pragma unroll
      for (int h = 1; h < H; ++h)
        *reinterpret_cast<double2*>(rec + 22 + 2 * h) = double2{v[9 + h], s[9 + h]};
      wave_lds_sync();
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (t >= nrj[j]) continue;
        double* r = lds + (16 * j + c) * RB;
        const double2 pl = *reinterpret_cast<const double2*>(r + 2 * g);
        const double2 pb = *reinterpret_cast<const double2*>(r + (g ? 12 + 2 * g : 0));
        const double2 R01 = *reinterpret_cast<const double2*>(r + 20);
        const double2 R23 = *reinterpret_cast<const double2*>(r + 22);
        double ch[4], dc[4];
        ch[0] = pl.x;
        dc[0] = pl.y;
#pragma unroll
        for (int q = 1; q < 4; ++q) {
          const double2 pp = *reinterpret_cast<const double2*>(r + 6 + 2 * q);
          ch[q] = pl.x * pp.x;
          dc[q] = fma(pl.y, pp.x, pl.x * pp.y);
        }
        d4 Y[H], Yd[H];
#pragma unroll
        for (int h = 0; h < H; ++h) {
          Y[h] = d4{0.0, 0.0, 0.0, 0.0};
          Yd[h] = d4{0.0, 0.0, 0.0, 0.0};
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int h = 0; h < H; ++h) {
            Y[h] = mfma_f64(dMa[j][h][q], ch[q], Y[h]);
            Yd[h] = mfma_f64(dMa[j][h][q], dc[q], Yd[h]);
          }
        const double R[4] = {R01.x, R01.y, R23.x, R23.y};
        double u[4], vs = 0.0;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          u[m] = pb.x * Y[0][m];
          vs = fma(R[m], fma(pb.y, Y[0][m], pb.x * Yd[0][m]), vs);
        }
#pragma unroll
        for (int h = 1; h < H; ++h) {
          const double2 ph = *reinterpret_cast<const double2*>(r + 22 + 2 * h);
          const double wh = pb.x * ph.x, wd = fma(pb.y, ph.x, pb.x * ph.y);
#pragma unroll
          for (int m = 0; m < 4; ++m) {
            u[m] = fma(wh, Y[h][m], u[m]);
            vs = fma(R[m], fma(wd, Y[h][m], wh * Yd[h][m]), vs);
          }
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) u[m] = add_xor32(add_xor16(u[m]));
        vs = add_xor32(add_xor16(vs));
        wave_lds_sync();
        r[g] = g == 0 ? u[0] : g == 1 ? u[1] : g == 2 ? u[2] : u[3];
        if (g == 0) r[4] = vs;
      }
      wave_lds_sync();
      if (live) {
        double nd[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) nd[m] = rec[m] * a.inv_nnei;
        // dx/dR_0 = dx/d(sw/r) std_0
        nd[0] = fma(rec[4] * a.inv_nnei * dxds, a.envp[pair * 8 + 4], nd[0]);
        double gv[3];
        env_grad(d[0], d[1], d[2], a.rcut_smth, a.rcut, a.inv_sw, isd, nd, gv);
        slot_out<AV>(a, ebase + slot, jatom, d, gv, own, reinterpret_cast<unsigned long long*>(rec));
      } else {
        rec[3] = __builtin_bit_cast(double, -1L);
      }
      wave_lds_sync();
      scatter_records<AV, RB>(a, lds, 64, lane);
    }
  }
  // slots outside the expansion's range (rare): the net and its slope
  bool any = __ballot(close) != 0;
  if constexpr (W > 1) any = __syncthreads_or(any);
  if (__builtin_expect(any && w == 0, 0)) {
    for (int j = 0; j < 4; ++j) {
      const int i = lane_int(q4.i, 16 * j);
      const double x0 = lane_double(xi, 16 * j), y0 = lane_double(yi, 16 * j),
                   z0 = lane_double(zi, 16 * j);
      if (!lane_int(q4.ok, 16 * j)) continue;
      const E* dTi = static_cast<const E*>(a.dT) + (long)i * 4 * L3;
      for (int tj = 0; tj < a.ntypes; ++tj) {
        const int pair = ti * a.ntypes + tj;
        const int nr = a.nreal[(long)i * a.ntypes + tj];
        const long ebase = (long)i * a.nnei + a.sec[tj];
        double avg[4], isd[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          avg[m] = a.envp[pair * 8 + m];
          isd[m] = 1.0 / a.envp[pair * 8 + 4 + m];
        }
        for (int t = 0; t < nr; t += 64) {
          double Rn[4], d[3] = {0.0, 0.0, 0.0}, y = 0.0;
          int k = 0;
          if (t + lane < nr) {
            k = a.nlist[ebase + t + lane];
            d[0] = a.ext[3L * k] - x0;
            d[1] = a.ext[3L * k + 1] - y0;
            d[2] = a.ext[3L * k + 2] - z0;
            y = env_row(a, d[0], d[1], d[2], avg, isd, Rn);
          }
          for (unsigned long long todo = __ballot(y > 1.0); todo; todo &= todo - 1) {
            const int src = __ffsll((long long)todo) - 1;
            double R[4], G[2], dG[2], nd[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) R[m] = lane_double(Rn[m], src);
            net_at<true>(a.nets + (long)pair * a.net_stride, a.emb, R[0], lds, lane, G, dG);
            double vs = 0.0;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
              double u = 0.0;
#pragma unroll
              for (int e = 0; e < 2; ++e) {
                const int f = lane + 64 * e;
                if (f >= L3) continue;
                const double dt = (double)dTi[m * L3 + f];
                u = fma(dt, G[e], u);
                vs = fma(R[m] * dt, dG[e], vs);
              }
              nd[m] = add_xor32(add_xor16(sum_c16(u))) * a.inv_nnei;
            }
            nd[0] += add_xor32(add_xor16(sum_c16(vs))) * a.inv_nnei;
            if (lane == src) {
              double gv[3], part[12];
#pragma unroll
              for (int q = 0; q < 12; ++q) part[q] = 0.0;
              env_grad(d[0], d[1], d[2], a.rcut_smth, a.rcut, a.inv_sw, isd, nd, gv);
              slot_out<AV>(a, ebase + t + lane, k, d, gv, part, reinterpret_cast<unsigned long long*>(lds));
#pragma unroll
              for (int q = 0; q < 12; ++q) lds[16 + q] = part[q];
            }
            wave_lds_sync();
            scatter_records<AV, RB>(a, lds, 1, lane);
            if (lane == 16 * j)
#pragma unroll
              for (int q = 0; q < 12; ++q) own[q] += lds[16 + q];
          }
        }
      }
    }
  }
  // the centre's own sums over the 16 lanes of its group
#pragma unroll
  for (int q = 0; q < 12; ++q) own[q] = sum_c16(own[q]);
  if constexpr (W > 1) {
    // ... and over the block's waves, in order
    __syncthreads();
    if (c == 0)
#pragma unroll
      for (int q = 0; q < 12; ++q) lds_all[(w * 4 + g) * 12 + q] = own[q];
    __syncthreads();
    if (w == 0 && c == 0)
#pragma unroll
      for (int q = 0; q < 12; ++q)
        for (int v = 1; v < W; ++v) own[q] += lds_all[(v * 4 + g) * 12 + q];
  }
  if (q4.ok && c == 0 && w == 0) {
    double* o = a.cpart + 12L * q4.i;
#pragma unroll
    for (int q = 0; q < 12; ++q) o[q] = own[q];
  }
}

namespace {
// Blocks of four waves up to this many groups of four centres (half a group
// per SIMD). Queued steps with blocks of one / four waves, us: water 192 atoms
// 177 / 147, 1536 338 / 314, 3993 440 / 442, 12288 861 / 975; Cu 864 262 / 236,
// 4000 461 / 462; HEA mixed 1024 262 / 232, 3456 489 / 528. With four groups of
// terms (a block's LDS then fills a compute unit) they cross a little lower, at
// about 430: water 1536 351 / 343, 2187 383 / 420; HEA mixed 1024 291 / 241, 2000
// 372 / 407, 2662 449 / 566.
constexpr int kSharedGroups = 512;

template <class K>
void run(K kern, hipStream_t st, const ExpandArgs& a, int nblock, int waves, size_t bytes) {
  DPAMD_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)bytes));
  hipLaunchKernelGGL(kern, dim3(nblock), dim3(64 * waves), bytes, st, a);
}
template <class E, int NU3, int H, int W>
void launch_w(hipStream_t st, const ExpandArgs& a, int nblock, bool bwd) {
  if (!bwd) run(k_expand_fwd<E, NU3, H, W>, st, a, nblock, W, sizeof(double) * W * fwd_lds(H));
  else if (a.vacc) run(k_expand_bwd<E, NU3, H, true, W>, st, a, nblock, W, sizeof(double) * W * bwd_lds(H));
  else run(k_expand_bwd<E, NU3, H, false, W>, st, a, nblock, W, sizeof(double) * W * bwd_lds(H));
}
template <class E, int NU3, int H>
void launch_g(hipStream_t st, const ExpandArgs& a, int ngroup, bool bwd) {
  if (ngroup <= kSharedGroups) launch_w<E, NU3, H, 4>(st, a, ngroup, bwd);
  else launch_w<E, NU3, H, 1>(st, a, ngroup, bwd);
}
template <class E, int NU3>
void launch_h(hipStream_t st, const ExpandArgs& a, int H, int ngroup, bool bwd) {
  H == 1 ? launch_g<E, NU3, 1>(st, a, ngroup, bwd)
         : H == 2 ? launch_g<E, NU3, 2>(st, a, ngroup, bwd) : launch_g<E, NU3, 4>(st, a, ngroup, bwd);
  DPAMD_LAUNCH_CHECK();
}
void launch_expand(hipStream_t st, const ExpandArgs& a, int H, bool f32, bool bwd) {
  const int nwave = a.wave_off[a.ntypes];
  if (nwave <= 0) return;
  const bool wide = a.emb[2] > 112;
  if (f32) {
    wide ? launch_h<float, 8>(st, a, H, nwave, bwd) : launch_h<float, 7>(st, a, H, nwave, bwd);
  } else {
    wide ? launch_h<double, 8>(st, a, H, nwave, bwd) : launch_h<double, 7>(st, a, H, nwave, bwd);
  }
}
}  // namespace

void launch_expand_fwd(hipStream_t st, const ExpandArgs& a, int H, bool f32) {
  launch_expand(st, a, H, f32, false);
}
void launch_expand_bwd(hipStream_t st, const ExpandArgs& a, int H, bool f32) {
  launch_expand(st, a, H, f32, true);
}

}  // namespace dpamd
