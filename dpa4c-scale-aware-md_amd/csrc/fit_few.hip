// Fitting net for few atoms (axis 16): forward, energy head, input gradient
// and dE/dT of every centre type in seven launches.
//
// With a few hundred rows the tiled GEMMs of fitting.hip are bound by latency:
// a layer's block walks its K loop in 16-wide chunks, each a global load, an
// LDS store and a barrier behind the last, about 1 us a chunk, while most of
// the chip idles (192 water atoms: 16-22 us a launch, one launch per layer
// and type, on forked streams). Here a block computes one tile of 16 or 32 rows x 16
// columns and its waves split K between them, so the loads of a wave's whole
// share are in flight at once and nothing waits on a barrier before the one
// that sums the waves' partials (in wave order); the types share a launch.
// The operands come straight from L2. The grids' x is the column tile, a
// multiple of the eight XCDs (blocks are dealt to them round robin), so each
// XCD reads its own eighth of the weights (2-4 MB a type, all of which every
// XCD would fetch otherwise) for all rows.
//
// The layers' epilogues are those of fitting.hip (reference semantics:
// h = act(xW+b) (+ residual), e = h.w_head + b_head + bias_atom_e[type],
// deepmd-op/overlays/op/pt/graph_fitting.cu:1-25, :614-719). T is double
// (FP64 MFMA) or float (fp32 MFMA, fp32 accumulation).
#include "fastmath.h"
#include "kernels.h"

namespace dpamd {

namespace {

constexpr int kU = 16;  // k-steps (of 4) whose operands are in flight at once

// The block's row tile: net, first row within the type, bucket position of it.
struct Tile {
  int t, row0, rows;
  long pos0;
};
template <class T>
__device__ __forceinline__ Tile find_tile(const FewArgs<T>& a, int block) {
  int t = 0;
  while (t + 1 < a.nt && block >= a.net[t + 1].tile0) ++t;
  const int row0 = a.tile_rows * (block - a.net[t].tile0);
  return Tile{t, row0, a.net[t].rows, (long)a.net[t].pos0 + row0};
}

// A tile's accumulator: fp64, or fp32 partial sums of at most 64 products
// added up in fp64 (flush), which leaves no more rounding than the bf16
// three-piece products of the general kernels (whose fp32 accumulators run
// over all of K): without it the forces of small mixed systems were 12 % further
// from their fp64 values than with those.
template <class T>
struct TileAcc {
  d4 s = d4{0.0, 0.0, 0.0, 0.0};
  __device__ __forceinline__ void add(double a, double b) { s = mfma(a, b, s); }
  __device__ __forceinline__ void flush() {}
};
template <>
struct TileAcc<float> {
  d4 s = d4{0.0, 0.0, 0.0, 0.0};
  f4 part = f4{0.0f, 0.0f, 0.0f, 0.0f};
  __device__ __forceinline__ void add(float a, float b) { part = mfma(a, b, part); }
  __device__ __forceinline__ void flush() {
#pragma unroll
    for (int r = 0; r < 4; ++r) s[r] += (double)part[r];
    part = f4{0.0f, 0.0f, 0.0f, 0.0f};
  }
};

// The waves' partial tiles (RT times 16 rows x 16 columns) in LDS; element
// (row, col) is then their sum in wave order.
template <class T, int RT>
__device__ __forceinline__ void park(double (*red)[16 * RT][17], const TileAcc<T> (&acc)[RT], int w,
                                     int g, int c) {
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[w][16 * t + Frag<T>::row(g, r)][c] = acc[t].s[r];
  __syncthreads();
}
template <class T, int NW, int RT>
__device__ __forceinline__ T sum_waves(double (*red)[16 * RT][17], int row, int col, T bias = T(0)) {
  double s = red[0][row][col];
#pragma unroll
  for (int k = 1; k < NW; ++k) s += red[k][row][col];
  return (T)(s + bias);
}

__device__ __forceinline__ double act(double x) { return tanh_fast(x); }
__device__ __forceinline__ float act(float x) { return tanh_f32(x); }

// First layer: H0 = tanh(D W0 + b0), D[16a + b] = sum_m T[m][a] T[m][b] formed
// in the A operand (lane (g, c): row c, b = 4q + g). Eight waves share the
// columns a.
constexpr int kFirstWaves = 8;
template <class T, int RT>
__global__ __launch_bounds__(64 * kFirstWaves) void k_few_first(FewArgs<T> a) {
  __shared__ double red[kFirstWaves][16 * RT][17];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const Tile tl = find_tile(a, blockIdx.y);
  const FewNet<T>& net = a.net[tl.t];
  const int N = a.F[0], col0 = 16 * blockIdx.x;
  if (col0 >= N) return;
  const T* Tr[RT];
  Vec4<T> tb[RT][4];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    Tr[t] = a.Tt + 4 * (tl.pos0 + min(16 * t + c, tl.rows - 1 - tl.row0));
#pragma unroll
    for (int q = 0; q < 4; ++q)
      tb[t][q] = *reinterpret_cast<const Vec4<T>*>(Tr[t] + (4 * q + g) * a.ldt);
  }
  const int per = (a.L3 + kFirstWaves - 1) / kFirstWaves;
  const int a0 = w * per, a1 = min(a.L3, a0 + per);
  const T* W = net.W[0] + (long)g * N + col0 + c;
  TileAcc<T> acc[RT];
  constexpr int U = RT > 1 ? 2 : 4;  // columns a (four k-steps each) in flight
  for (int k = a0; k < a1; k += U) {
    Vec4<T> ta[U][RT];
    T b[U][4];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int ak = min(k + u, a1 - 1);
#pragma unroll
      for (int t = 0; t < RT; ++t) ta[u][t] = *reinterpret_cast<const Vec4<T>*>(Tr[t] + ak * a.ldt);
#pragma unroll
      for (int q = 0; q < 4; ++q) b[u][q] = W[(long)(16 * ak + 4 * q) * N];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k + u >= a1) break;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          const Vec4<T>&x = ta[u][t], &y = tb[t][q];
          acc[t].add(x.x * y.x + x.y * y.y + x.z * y.z + x.w * y.w, b[u][q]);
        }
    }
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t].flush();
  }
  park<T, RT>(red, acc, w, g, c);
  const int col = col0 + (threadIdx.x & 15);
  for (int row = threadIdx.x >> 4; row < 16 * RT; row += 4 * kFirstWaves)
    if (tl.row0 + row < tl.rows)
      a.H0[(tl.pos0 + row) * N + col] =
          act(sum_waves<T, kFirstWaves, RT>(red, row, threadIdx.x & 15, net.b[0][col]));
}

// The other layers, four waves a block. STAGE 1: H1 = [H0] + idt1 t, t =
// tanh(H0 W1 + b1). STAGE 2: the last layer with the energy head: dZ2 = Wo
// idt2 (1 - t^2) and the row's partial energy over the block's columns.
// STAGE 3: dH1 = [Wo] + dZ2 W2^T, dZ1 = dH1 idt1 (1 - T1^2), and (first
// column tile) the atom energies. STAGE 4: dH0 = [dH1] + dZ1 W1^T, dZ0 = dH0
// (1 - H0^2). ([.]: on square layers.)
template <class T, int STAGE, int RT>
__global__ __launch_bounds__(256) void k_few_layer(FewArgs<T> a) {
  __shared__ double red[4][16 * RT][17];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const Tile tl = find_tile(a, blockIdx.y);
  const FewNet<T>& net = a.net[tl.t];
  const int K = STAGE == 1 ? a.F[0] : STAGE == 2 ? a.F[1] : STAGE == 3 ? a.F[2] : a.F[1];
  const int N = STAGE == 1 ? a.F[1] : STAGE == 2 ? a.F[2] : STAGE == 3 ? a.F[1] : a.F[0];
  const T* A = STAGE == 1 ? a.H0 : STAGE == 2 ? a.H1 : STAGE == 3 ? a.dZa : a.dZb;
  const T* W = STAGE == 1 ? net.W[1] : STAGE == 2 ? net.W[2] : STAGE == 3 ? net.WT[2] : net.WT[1];
  const int col0 = 16 * blockIdx.x;
  if (col0 >= N) return;
  const int per = K / 16;  // k-steps of one wave (K % 16 == 0)
  const int k0 = 4 * per * w + g;
  const T* Ar[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
    Ar[t] = A + (tl.pos0 + min(16 * t + c, tl.rows - 1 - tl.row0)) * K + k0;
  const T* Br = W + (long)k0 * N + col0 + c;
  // the epilogue's inputs, read ahead of the products: the summand (forward the
  // bias, backward the residual's gradient), the layer's input or activation,
  // and the column's parameters
  const int col = col0 + (threadIdx.x & 15);
  T add[RT], in[RT];
  const T id = STAGE == 1 || STAGE == 3 ? (net.idt[1] ? net.idt[1][col] : T(1))
               : STAGE == 2             ? (net.idt[2] ? net.idt[2][col] : T(1))
                                        : T(1);
  const T wo = STAGE == 2 || (STAGE == 3 && net.idt[2]) ? net.Wo[col] : T(0);
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int row = min(16 * t + (int)(threadIdx.x >> 4), tl.rows - 1 - tl.row0);
    const long o = (tl.pos0 + row) * N + col;
    add[t] = STAGE <= 2 ? net.b[STAGE <= 2 ? STAGE : 0][col]
             : STAGE == 3 ? wo
             : net.idt[1] ? a.dH[o] : T(0);
    in[t] = STAGE == 1 ? (net.idt[1] ? a.H0[o] : T(0))
            : STAGE == 2 ? (net.idt[2] ? a.H1[o] : T(0))
            : STAGE == 3 ? a.T1[o] : a.H0[o];
  }
  TileAcc<T> acc[RT];
  for (int q0 = 0; q0 < per; q0 += kU) {
    T av[kU][RT], bv[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int q = min(q0 + u, per - 1);
#pragma unroll
      for (int t = 0; t < RT; ++t) av[u][t] = Ar[t][4 * q];
      bv[u] = Br[4L * N * q];
    }
#pragma unroll
    for (int u = 0; u < kU; ++u)
      if (q0 + u < per)
#pragma unroll
        for (int t = 0; t < RT; ++t) acc[t].add(av[u][t], bv[u]);
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t].flush();
  }
  park<T, RT>(red, acc, w, g, c);
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int row = 16 * t + (threadIdx.x >> 4);
    const T z = sum_waves<T, 4, RT>(red, row, threadIdx.x & 15, add[t]);
    const bool ok = tl.row0 + row < tl.rows;
    const long R = tl.pos0 + row, o = R * N + col;
    if constexpr (STAGE == 1) {
      if (ok) {
        const T th = act(z);
        a.T1[o] = th;
        a.H1[o] = in[t] + id * th;  // (not square: 0 + 1 th)
      }
    } else if constexpr (STAGE == 2) {
      double e = 0.0;
      if (ok) {
        const T th = act(z);
        const T h = in[t] + id * th;
        a.dZa[o] = wo * id * (T(1) - th * th);
        e = (double)h * (double)wo;
      }
#pragma unroll
      for (int off = 8; off > 0; off >>= 1) e += shfl_xor_d(e, off);
      if (ok && (threadIdx.x & 15) == 0) a.epart[R * (N / 16) + blockIdx.x] = e;
    } else if constexpr (STAGE == 3) {
      if (ok) {
        a.dH[o] = z;
        a.dZb[o] = z * id * (T(1) - in[t] * in[t]);
        if (blockIdx.x == 0 && (threadIdx.x & 15) == 0) {
          const int nc = a.F[2] / 16;
          double e = 0.0;
          for (int k = 0; k < nc; ++k) e += a.epart[R * nc + k];
          a.e[R] = e + net.bo + net.bias;
        }
      }
    } else {
      if (ok) a.dZa[o] = z * (T(1) - in[t] * in[t]);
    }
  }
}

// dE/dD = dZ0 W0^T of a row tile and eight columns a (two per wave), computed
// transposed (D'[b][row]: register r of lane (g, c) is dD[row c][a][b =
// row(g, r)]) and contracted at once:
//   dT[m][a] = sum_b dD[a][b] T[m][b] (stored; a < 16: to ws, slice
//   a.slices), and the block's share of sum_a dD[a][b] T[m][a] (b < 16) to
//   ws slice blockIdx.x; k_few_combine adds the slices in order.
constexpr int kDtCols = 8;
template <class T, int RT>
__global__ __launch_bounds__(256) void k_few_dT(FewArgs<T> a) {
  extern __shared__ __align__(16) char few_lds[];
  T* Z = reinterpret_cast<T*>(few_lds);  // [16 RT][K + 4], then [4 waves][16 rows][64]
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const Tile tl = find_tile(a, blockIdx.y);
  const FewNet<T>& net = a.net[tl.t];
  const int K = a.F[0], LD = K + 4, nq = K / 4, Dn = 16 * a.L3;
  if ((int)blockIdx.x >= a.slices) return;
  // dZ0 rows: 16 threads a row, eight loads in flight
  for (int t = 0; t < RT; ++t) {
    const int r = 16 * t + (threadIdx.x >> 4), k0 = threadIdx.x & 15;
    const bool in = tl.row0 + r < tl.rows;
    const T* src = a.dZa + (tl.pos0 + (in ? r : 0)) * K;
    for (int k = k0; k < K; k += 128) {
      T v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = src[min(k + 16 * u, K - 1)];
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (k + 16 * u < K) Z[r * LD + k + 16 * u] = in ? v[u] : T(0);
    }
  }
  const T* Tr[RT];
  Vec4<T> tb[RT][4];
  int atom[RT];
  T acc2[RT][4][4];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int row = 16 * t + c;
    Tr[t] = a.Tt + 4 * (tl.pos0 + min(row, tl.rows - 1 - tl.row0));
    atom[t] = tl.row0 + row < tl.rows ? a.items[tl.pos0 + row] : -1;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      tb[t][r] = *reinterpret_cast<const Vec4<T>*>(Tr[t] + Frag<T>::row(g, r) * a.ldt);
#pragma unroll
      for (int m = 0; m < 4; ++m) acc2[t][r][m] = T(0);
    }
  }
  const T* Zr = Z + c * LD + g;
  const int col0 = kDtCols * blockIdx.x + 2 * w, ncol = min(2, a.L3 - col0);
  TileAcc<T> acc[RT];
  Vec4<T> ta[RT];
  // step: kU k-steps of column col0 + step / chunks; W0^T[k][16 col + c]
  const int chunks = (nq + kU - 1) / kU, steps = ncol > 0 ? ncol * chunks : 0;
  auto load = [&](T (&wv)[kU], int step) {
    const int e = min(step, steps - 1) / chunks, q0 = kU * (min(step, steps - 1) - e * chunks);
    const T* Wr = net.WT[0] + (long)g * Dn + 16 * (col0 + e) + c;
#pragma unroll
    for (int u = 0; u < kU; ++u) wv[u] = Wr[4L * Dn * min(q0 + u, nq - 1)];
  };
  auto multiply = [&](const T (&wv)[kU], int step) {
    if (step >= steps) return;
    const int e = step / chunks, q0 = kU * (step - e * chunks), col = col0 + e;
    if (q0 == 0) {
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        acc[t] = TileAcc<T>{};
        ta[t] = *reinterpret_cast<const Vec4<T>*>(Tr[t] + col * a.ldt);
      }
    }
    // (four k-steps' rows are read ahead of their products)
    T z[2][4][RT];
    auto rows = [&](T (&zz)[4][RT], int u0) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int t = 0; t < RT; ++t) zz[u][t] = Zr[16 * t * LD + 4 * min(q0 + u0 + u, nq - 1)];
    };
    rows(z[0], 0);
#pragma unroll
    for (int u0 = 0; u0 < kU; u0 += 4) {
      if (u0 + 4 < kU) rows(z[(u0 / 4 + 1) & 1], u0 + 4);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (q0 + u0 + u < nq)
#pragma unroll
          for (int t = 0; t < RT; ++t) acc[t].add(wv[u0 + u], z[(u0 / 4) & 1][u][t]);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t].flush();
    if (q0 + kU < nq) return;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      const T tm[4] = {ta[t].x, ta[t].y, ta[t].z, ta[t].w};
      double s[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        double v = 0.0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const Vec4<T>& y = tb[t][r];
          v += acc[t].s[r] * (double)(m == 0 ? y.x : m == 1 ? y.y : m == 2 ? y.z : y.w);
          acc2[t][r][m] += (T)acc[t].s[r] * tm[m];
        }
        s[m] = add_xor32(add_xor16(v));
      }
      const double mine = g == 0 ? s[0] : g == 1 ? s[1] : g == 2 ? s[2] : s[3];
      const long pos = tl.pos0 + 16 * t + c;
      if (atom[t] >= 0) {
        if (col >= 16) a.dT[((long)atom[t] * 4 + g) * a.L3 + col] = (T)mine;
        else a.ws[((long)a.slices * a.nb + pos) * 64 + 16 * g + col] = mine;
        if (a.dD)
#pragma unroll
          for (int r = 0; r < 4; ++r) a.dD[pos * Dn + 16 * col + Frag<T>::row(g, r)] = (T)acc[t].s[r];
      }
    }
  };
  if (steps > 0) {
    T w0[kU], w1[kU], w2[kU];
    load(w0, 0);
    load(w1, 1);
    __syncthreads();
    for (int k = 0; k < steps; k += 3) {
      load(w2, k + 2);
      multiply(w0, k);
      load(w0, k + 3);
      multiply(w1, k + 1);
      load(w1, k + 4);
      multiply(w2, k + 2);
    }
  } else {
    __syncthreads();
  }
  // the block's second-term share, summed over its waves in order
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int m = 0; m < 4; ++m) Z[(w * 16 + c) * 64 + 16 * m + Frag<T>::row(g, r)] = acc2[t][r][m];
    __syncthreads();
    for (int q = threadIdx.x; q < 16 * 64; q += 256) {
      const int r = 16 * t + (q >> 6);
      if (tl.row0 + r >= tl.rows) continue;
      const double s = (((double)Z[q] + (double)Z[1024 + q]) + (double)Z[2048 + q]) + (double)Z[3072 + q];
      a.ws[((long)blockIdx.x * a.nb + tl.pos0 + r) * 64 + (q & 63)] = s;
    }
  }
}

// dT[.][m][b < 16]: the first term plus the second term's slices in order
template <class T>
__global__ __launch_bounds__(256) void k_few_combine(FewArgs<T> a) {
  const long q = (long)blockIdx.x * 256 + threadIdx.x;
  if (q >= 64L * a.nb) return;
  double s = 0.0;
  for (int k = 0; k < a.slices; ++k) s += a.ws[64L * k * a.nb + q];
  const int e = (int)(q & 63);
  a.dT[((long)a.items[q >> 6] * 4 + (e >> 4)) * a.L3 + (e & 15)] =
      (T)(a.ws[64L * a.slices * a.nb + q] + s);
}

}  // namespace

int few_slices(int L3) { return (L3 + kDtCols - 1) / kDtCols; }

// Rows of a block: two row tiles share each weight fragment once the tiles
// alone fill the device.
int few_tile_rows(int nb) { return nb > 384 ? 32 : 16; }

size_t few_lds_bytes(int nb, int F0, size_t esize) {
  return esize * std::max(few_tile_rows(nb) * (F0 + 4), 4 * 16 * 64);
}

namespace {
template <class T, int RT>
void run_few(hipStream_t st, const FewArgs<T>& a, int tiles) {
  // grids: columns (padded to a multiple of the XCDs) x row tiles
  auto cols = [&](int n) { return dim3((n + kXcds - 1) / kXcds * kXcds, tiles); };
  hipLaunchKernelGGL((k_few_first<T, RT>), cols(a.F[0] / 16), dim3(64 * kFirstWaves), 0, st, a);
  DPAMD_LAUNCH_CHECK();
  hipLaunchKernelGGL((k_few_layer<T, 1, RT>), cols(a.F[1] / 16), dim3(256), 0, st, a);
  DPAMD_LAUNCH_CHECK();
  hipLaunchKernelGGL((k_few_layer<T, 2, RT>), cols(a.F[2] / 16), dim3(256), 0, st, a);
  DPAMD_LAUNCH_CHECK();
  hipLaunchKernelGGL((k_few_layer<T, 3, RT>), cols(a.F[1] / 16), dim3(256), 0, st, a);
  DPAMD_LAUNCH_CHECK();
  hipLaunchKernelGGL((k_few_layer<T, 4, RT>), cols(a.F[0] / 16), dim3(256), 0, st, a);
  DPAMD_LAUNCH_CHECK();
  hipLaunchKernelGGL((k_few_dT<T, RT>), cols(a.slices), dim3(256),
                     few_lds_bytes(a.nb, a.F[0], sizeof(T)), st, a);
  DPAMD_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_few_combine<T>, dim3((unsigned)((64L * a.nb + 255) / 256)), dim3(256), 0, st, a);
  DPAMD_LAUNCH_CHECK();
}
}  // namespace

template <class T>
void launch_fitting_few(hipStream_t st, const FewArgs<T>& a) {
  int tiles = 0;
  for (int t = 0; t < a.nt; ++t)
    tiles = std::max(tiles, a.net[t].tile0 + (a.net[t].rows + a.tile_rows - 1) / a.tile_rows);
  if (tiles == 0) return;
  a.tile_rows == 16 ? run_few<T, 1>(st, a, tiles) : run_few<T, 2>(st, a, tiles);
}

template void launch_fitting_few<double>(hipStream_t, const FewArgs<double>&);
template void launch_fitting_few<float>(hipStream_t, const FewArgs<float>&);

}  // namespace dpamd
