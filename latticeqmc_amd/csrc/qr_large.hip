// Pre-pivoted Householder QR of matrices above 256 (up to QL_NMAX) over several workgroups each.
//
// The column order (decreasing norm) is found and applied first (k_ql_norms, k_ql_order,
// k_ql_gather: A = W P).  Then one launch per 16-column panel p (k_ql_step): workgroup 0 of a
// matrix applies panel p - 1 to panel p's columns and factors it, while the others apply panel
// p - 1 to 32 columns each of the rest, so the dependent column steps of a factorisation run
// beside the update.  D^-1 R goes over W at the end (k_ql_out), and Q is formed 32 columns per
// workgroup, held in registers, from the last panel to the first (k_ql_formq).
//
// A 512-thread workgroup holds a column block with wavefront w keeping the row tiles t = w, w + 8,
// ... in the accumulator layout of the FP64 matrix cores (row 16 t + l / 16 + 4 v, column l % 16 of
// lane l), which is the operand layout of V^T X; the eight partial products meet in LDS.  X is
// read and written once per panel.
//
// Bound by the chain of 16 column steps per panel (one workgroup barrier each: 28 us for the panel
// alone, 55 us on average with the update beside it at N = 576, 64 matrices) and by traffic to the
// trailing matrices of the first panels; Q formation by the two barriers per panel.  64 matrices of
// 576: factorisation 10.15 -> 2.17 ms, Q 2.66 -> 0.75 ms against the one-workgroup kernels
// (k_qr_blocked, k_qr_formq), which stream the trailing matrix through one compute unit between
// wavefront-serial panels.  Reading V once and transposing its tiles in LDS, with the next panel's
// fetched during the update, took Q from 1.18 to 0.75 ms.
#include "common.h"

#include <algorithm>

namespace lqmc {

typedef double ql_v4d __attribute__((ext_vector_type(4)));

constexpr int QL_THREADS = 512;
constexpr int QL_WAVES = 8;
constexpr int QL_SLOTS = 5;                      // row tiles per wavefront
constexpr int QL_NMAX = 16 * QL_WAVES * QL_SLOTS;  // 640

__device__ inline ql_v4d ql_mma(double a, double b, ql_v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

__device__ inline void ql_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ inline double ql_readlane(double v, int l) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// v summed over the lanes l, l ^ 16, l ^ 32, l ^ 48 (one column of an accumulator tile).
__device__ inline double ql_colsum(double v) {
  auto halves = [](unsigned long long a, unsigned long long b, auto swap) {
    const auto l = swap((unsigned)a, (unsigned)b);
    const auto h = swap((unsigned)(a >> 32), (unsigned)(b >> 32));
    const double x = __longlong_as_double((long long)(((unsigned long long)h[0] << 32) | l[0]));
    const double y = __longlong_as_double((long long)(((unsigned long long)h[1] << 32) | l[1]));
    return x + y;
  };
  unsigned long long b = (unsigned long long)__double_as_longlong(v);
  v = halves(b, b, [](unsigned x, unsigned y) { return __builtin_amdgcn_permlane32_swap(x, y, false, false); });
  b = (unsigned long long)__double_as_longlong(v);
  return halves(b, b, [](unsigned x, unsigned y) { return __builtin_amdgcn_permlane16_swap(x, y, false, false); });
}

// 1 / x and 1 / sqrt(x) (x well inside the exponent range) by Newton steps from the hardware estimates.
__device__ inline double ql_rcp(double x) {
#ifdef LQMC_CPU_EMU
  return 1.0 / x;
#else
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
#endif
}
__device__ inline double ql_rsqrt(double x) {
#ifdef LQMC_CPU_EMU
  return 1.0 / sqrt(x);
#else
  double r = __builtin_amdgcn_rsq(x);
  double e = fma(-x * r, r, 1.0);
  r = fma(r * e, fma(e, 0.375, 0.5), r);
  e = fma(-x * r, r, 1.0);
  return fma(r * e, 0.5, r);
#endif
}

// Scratch of a task: the squared column norms in D (free until panel 0 is factored), the column
// order in Q (free until Q is formed).
__device__ inline double* ql_norms(const QrTask& tk) { return tk.D; }
__device__ inline int* ql_order(const QrTask& tk) { return reinterpret_cast<int*>(tk.Q); }

// ---- column order ---------------------------------------------------------------------------------
// Squared norms of 64 columns: four row groups of one wavefront each, combined in order.
__global__ __launch_bounds__(256) void k_ql_norms(const QrTask* __restrict__ tasks, int nblk, ChainState* st) {
  const QrTask tk = tasks[blockIdx.x / nblk];
  const int N = tk.N, lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int c0 = 64 * (blockIdx.x % nblk), c = c0 + lane;
  if (c0 >= N) return;
  LQMC_DYNAMIC_LDS(double, sm);  // [4][64]
  double s = 0.0;
  if (c < N)
    for (int r0 = g; r0 < N; r0 += 64) {  // 16 loads in flight, summed in row order
      double x[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) x[u] = ldg0(gptr(tk.W), (size_t)(r0 + 4 * u) * N + c, r0 + 4 * u < N);
#pragma unroll
      for (int u = 0; u < 16; ++u) s = fma(x[u], x[u], s);
    }
  sm[threadIdx.x] = s;
  __syncthreads();
  if (g == 0 && c < N) {
    s = (sm[lane] + sm[64 + lane]) + (sm[128 + lane] + sm[192 + lane]);
    if (!(s >= 0.0)) {  // a NaN: last in the order
      s = -1.0;
      if (st) atomicOr(&st[tk.chain].flags, 8u);
    }
    ql_norms(tk)[c] = s;
  }
}

// Ranks of 64 columns by decreasing norm, ties by index (four wavefronts share the comparisons).
__global__ __launch_bounds__(256) void k_ql_order(const QrTask* __restrict__ tasks, int nblk) {
  const QrTask tk = tasks[blockIdx.x / nblk];
  const int N = tk.N, lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int c0 = 64 * (blockIdx.x % nblk), c = c0 + lane;
  if (c0 >= N) return;
  LQMC_DYNAMIC_LDS(double, sm);
  double* norms = sm;                                   // [N]
  int* rk = reinterpret_cast<int*>(norms + QL_NMAX);    // [4][64]
  for (int i = threadIdx.x; i < N; i += 256) norms[i] = ql_norms(tk)[i];
  __syncthreads();
  const double nc = norms[c < N ? c : 0];
  int rank = 0;
#pragma unroll 8
  for (int k = g; k < N; k += 4) {
    const double n2 = norms[k];
    rank += (n2 > nc) || (n2 == nc && k < c);
  }
  rk[threadIdx.x] = rank;
  __syncthreads();
  if (g == 0 && c < N) {
    rank = (rk[lane] + rk[64 + lane]) + (rk[128 + lane] + rk[192 + lane]);
    ql_order(tk)[rank] = c;
    if (tk.perm) tk.perm[rank] = c;
  }
}

constexpr int QL_ROWS = 8;  // rows per workgroup of the two permuting copies

// A = W P, eight rows per workgroup through LDS.
__global__ __launch_bounds__(256) void k_ql_gather(const QrTask* __restrict__ tasks, int nblk) {
  const QrTask tk = tasks[blockIdx.x / nblk];
  const int N = tk.N, r0 = QL_ROWS * (blockIdx.x % nblk);
  if (r0 >= N) return;
  const int nr = min(QL_ROWS, N - r0);
  LQMC_DYNAMIC_LDS(double, sm);  // [nr][N]
  const LQMC_GLOBAL double* W = gptr(tk.W) + (size_t)r0 * N;
  LQMC_GLOBAL double* A = gptr(tk.A) + (size_t)r0 * N;
  const int* ord = ql_order(tk);
  for (int e = threadIdx.x; e < nr * N; e += 256) sm[e] = W[e];
  __syncthreads();
  for (int c = threadIdx.x; c < N; c += 256) {
    const int pc = ord[c];
    for (int r = 0; r < nr; ++r) A[r * N + c] = sm[r * N + pc];
  }
}

// V'' = D^-1 R P^T (columns to their original places) or R' = D^-1 R over W, R in A's upper triangle.
__global__ __launch_bounds__(256) void k_ql_out(const QrTask* __restrict__ tasks, int nblk) {
  const QrTask tk = tasks[blockIdx.x / nblk];
  const int N = tk.N, r0 = QL_ROWS * (blockIdx.x % nblk);
  if (r0 >= N) return;
  const int nr = min(QL_ROWS, N - r0);
  LQMC_DYNAMIC_LDS(double, sm);  // [nr][N]
  LQMC_GLOBAL double* W = gptr(tk.W) + (size_t)r0 * N;
  const LQMC_GLOBAL double* A = gptr(tk.A) + (size_t)r0 * N;
  const int* ord = ql_order(tk);
  for (int c = threadIdx.x; c < N; c += 256) {
    const int pc = tk.perm ? c : ord[c];
    for (int r = 0; r < nr; ++r) sm[r * N + pc] = c >= r0 + r ? A[r * N + c] / tk.D[r0 + r] : 0.0;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < nr * N; e += 256) W[e] = sm[e];
}

// ---- block reflectors ------------------------------------------------------------------------------
// This wavefront's part of a column block: NC 16-column tiles of its row tiles.
template <int NC>
using QlBlock = ql_v4d[QL_SLOTS][NC];

// A panel's V in this wavefront's row tiles (below the diagonal of A, explicit unit diagonal) and T
// (TRANS: T^T), both as left operands of products over rows.
struct QlV {
  double va[QL_SLOTS][4], tt[4];
};

template <bool TRANS>
__device__ __attribute__((always_inline)) inline void ql_load_v(QlV& p, const QrTask& tk, int P) {
  const int N = tk.N, lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readlane((int)threadIdx.x >> 6, 0);
  const int ca = 16 * P + li;
  const unsigned lane_off = lk * N + ca;  // the rest of an address is uniform
#pragma unroll
  for (int i = 0; i < QL_SLOTS; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r0 = 16 * (QL_WAVES * i + wave) + 4 * v, ra = r0 + lk;
      p.va[i][v] = ldg0(gptr(tk.A) + (size_t)min(r0, N - 1) * N, lane_off, ra < N && ra > ca);
    }
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int q = 4 * s + lk;
    p.tt[s] = gptr(tk.Tt)[(size_t)P * 256 + (TRANS ? q * 16 + li : li * 16 + q)];
  }
}

// X <- (I - V T' V^T) X for panel P's V and T' = T^T (TRANS) or T, on a column block spread over the
// workgroup.  wp: [8][NC][64][4] doubles of partial products; tb: [8][16][17], where each wavefront
// transposes its tiles of V (read from memory in that order they come as 32-byte pieces).  Row tiles
// above the panel and past the matrix are skipped.  The V of panel next is fetched during the update
// (next < 0: none).  Two barriers.
constexpr int QL_TB = 16 * 17;
template <int NC, bool TRANS>
__device__ __attribute__((always_inline)) inline void ql_apply(QlBlock<NC>& acc, QlV& p, const QrTask& tk, int P,
                                                               int next, double* wp, double* tb) {
  const int N = tk.N, lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readlane((int)threadIdx.x >> 6, 0);
  tb += wave * QL_TB;
  double vb[QL_SLOTS][4], tt[4];
  ql_v4d w[NC];
#pragma unroll
  for (int n = 0; n < NC; ++n) w[n] = ql_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int s = 0; s < 4; ++s) tt[s] = p.tt[s];
#pragma unroll
  for (int i = 0; i < QL_SLOTS; ++i) {
    const int t = QL_WAVES * i + wave;
    if (!TRANS && (t < P || 16 * t >= N)) continue;
    ql_wave_sync();
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int q = lk + 4 * v;
      const double a = t == P && q == li ? 1.0 : p.va[i][v];
      tb[q * 17 + li] = a;
#pragma unroll
      for (int n = 0; n < NC; ++n) w[n] = ql_mma(a, acc[i][n][v], w[n]);
    }
    ql_wave_sync();
#pragma unroll
    for (int v = 0; v < 4; ++v) vb[i][v] = -tb[li * 17 + lk + 4 * v];
  }
#pragma unroll
  for (int n = 0; n < NC; ++n) *reinterpret_cast<ql_v4d*>(wp + ((wave * NC + n) * 64 + lane) * 4) = w[n];
  if (next >= 0) ql_load_v<TRANS>(p, tk, next);
  __syncthreads();
  ql_v4d w2[NC];
#pragma unroll
  for (int n = 0; n < NC; ++n) {
    ql_v4d s = *reinterpret_cast<const ql_v4d*>(wp + (n * 64 + lane) * 4);
#pragma unroll
    for (int u = 1; u < QL_WAVES; ++u) s = s + *reinterpret_cast<const ql_v4d*>(wp + ((u * NC + n) * 64 + lane) * 4);
    w2[n] = ql_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < 4; ++k) w2[n] = ql_mma(tt[k], s[k], w2[n]);
  }
  __syncthreads();  // wp is free again
#pragma unroll
  for (int i = 0; i < QL_SLOTS; ++i) {
    const int t = QL_WAVES * i + wave;
    if (!TRANS && (t < P || 16 * t >= N)) continue;
#pragma unroll
    for (int n = 0; n < NC; ++n)
#pragma unroll
      for (int k = 0; k < 4; ++k) acc[i][n] = ql_mma(vb[i][k], w2[n][k], acc[i][n]);
  }
}

// Columns c0 .. c0 + 16 NC - 1 of A from row tile P on (zero elsewhere), and back.
template <int NC>
__device__ __attribute__((always_inline)) inline void ql_load(QlBlock<NC>& acc, const QrTask& tk, int P, int c0) {
  const int N = tk.N, lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readlane((int)threadIdx.x >> 6, 0);
  const unsigned lane_off = lk * N + li;
#pragma unroll
  for (int i = 0; i < QL_SLOTS; ++i)
#pragma unroll
    for (int n = 0; n < NC; ++n)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int t = QL_WAVES * i + wave, r0 = 16 * t + 4 * v, c = c0 + 16 * n + li;
        acc[i][n][v] =
            ldg0(gptr(tk.A) + (size_t)min(r0, N - 1) * N, lane_off + c0 + 16 * n, t >= P && r0 + lk < N && c < N);
      }
}
template <int NC>
__device__ __attribute__((always_inline)) inline void ql_store(const QlBlock<NC>& acc, const QrTask& tk, int P,
                                                               int c0) {
  const int N = tk.N, lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readlane((int)threadIdx.x >> 6, 0);
  const unsigned lane_off = lk * N + li;
#pragma unroll
  for (int i = 0; i < QL_SLOTS; ++i)
#pragma unroll
    for (int n = 0; n < NC; ++n)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int t = QL_WAVES * i + wave, r0 = 16 * t + 4 * v, c = c0 + 16 * n + li;
        if (t >= P && r0 + lk < N && c < N) (gptr(tk.A) + (size_t)r0 * N + c0 + 16 * n)[lane_off] = acc[i][n][v];
      }
}

// ---- panel factorisation -----------------------------------------------------------------------------
struct QlShared {
  double* xb;    // [8][6][16] pivot column by tile, each wavefront its own rows (last: the diagonal tile)
  double* part;  // [2][8][16] partial products of either parity
  double* row;   // [2][16] row j of the panel
  double* rbuf;  // [16][16] the panel's rows of R
  double* zb;    // [16] V^T v_q in the order of QlPanel::tr
};
constexpr int QL_SHARED = QL_WAVES * (QL_SLOTS + 1) * 16 + 2 * QL_WAVES * 16 + 32 + 256 + 16;  // doubles

struct QlPanel {
  ql_v4d pt;   // copy of the diagonal tile (the wavefront that holds it)
  ql_v4d tr;   // T[c][l / 16 + 4 i] (wavefront 0)
  double scal, beta, tau;
  bool zero;
};

// Householder steps of columns 4 HV .. 4 HV + 3 (below w): lane l holds column l % 16.  The pivot
// column reaches the lanes of the other columns through LDS (a wavefront needs its own rows only),
// x^T col of every column is one multiply-add per element, a sum over four lanes and one over the
// wavefronts (the barrier).  With u = x - beta e_j, beta = -sign(alpha) |x|:
//   col -= u (u^T col) / (|x| (|x| + |alpha|));
// a column of V stays u's tail, unscaled, until the panel is done.  The same products with the
// columns left of q are V^T v_q, which give column q of T: T[:, q] = -tau T (V^T v_q).
template <int HV>
__device__ __attribute__((always_inline)) inline void ql_columns(QlBlock<1>& acc, QlPanel& p, const QlShared& sh, int P,
                                                                 int w) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readlane((int)threadIdx.x >> 6, 0);
  const bool own = (P & (QL_WAVES - 1)) == wave;  // this wavefront holds the diagonal tile
  ql_v4d* xw = reinterpret_cast<ql_v4d*>(sh.xb) + wave * (QL_SLOTS + 1) * 4 + lk;
#pragma unroll 1
  for (int hk = 0; hk < 4; ++hk) {
    const int q = 4 * HV + hk, par = q & 1;
    if (q >= w) break;
    ql_wave_sync();  // the previous column's reads are done
    if (li == q) {
#pragma unroll
      for (int i = 0; i < QL_SLOTS; ++i) {
        ql_v4d m = acc[i][0];
        const int t = QL_WAVES * i + wave;
        if (t <= P) m = ql_v4d{0.0, 0.0, 0.0, 0.0};
        xw[4 * i] = m;
      }
      ql_v4d m;
#pragma unroll
      for (int v = 0; v < 4; ++v) m[v] = own && v >= HV && (v > HV || lk >= hk) ? p.pt[v] : 0.0;
      xw[4 * QL_SLOTS] = m;
    }
    ql_wave_sync();
    ql_v4d x[QL_SLOTS];
#pragma unroll
    for (int i = 0; i < QL_SLOTS; ++i) x[i] = xw[4 * i];
    const ql_v4d xd = xw[4 * QL_SLOTS];
    ql_v4d s = xd * p.pt;
#pragma unroll
    for (int i = 0; i < QL_SLOTS; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) s[v] = fma(x[i][v], acc[i][0][v], s[v]);
    const double yp = ql_colsum((s[0] + s[1]) + (s[2] + s[3]));
    if (lk == 0) sh.part[(par * QL_WAVES + wave) * 16 + li] = yp;
    if (own) {
      const double b = ql_colsum(lk == hk ? p.pt[HV] : 0.0);
      if (lk == 0) sh.row[par * 16 + li] = b;
    }
    __syncthreads();
    double y = 0.0;
#pragma unroll
    for (int u = 0; u < QL_WAVES; ++u) y += sh.part[(par * QL_WAVES + u) * 16 + li];
    const double bc = sh.row[par * 16 + li];
    const double nn = ql_readlane(y, q), alpha = ql_readlane(bc, q);
    const double r = ql_rsqrt(nn);
    double nrm = nn * r, h = nrm + fabs(alpha);
    double rden = ql_rcp(nrm * h), scal = nrm * rden;
    p.tau = h * r;
    if (__builtin_expect(!(nn > 1e-280 && nn < 1e280), 0)) {  // outside the estimates' range
      nrm = sqrt(nn > 0.0 ? nn : 0.0);
      if (nrm == 0.0) {
        rden = p.tau = scal = 0.0;
        p.zero = true;
      } else {
        h = nrm + fabs(alpha);
        rden = 1.0 / nrm / h;
        p.tau = h / nrm;
        scal = 1.0 / h;
      }
    }
    const double beta = alpha >= 0.0 ? -nrm : nrm;
    scal = alpha >= 0.0 ? scal : -scal;
    const double ut = fma(-beta, bc, y);  // u^T col (the columns left of q: u^T u_c)
    const double kap = li > q ? -(ut * rden) : 0.0;
#pragma unroll
    for (int v = HV; v < 4; ++v) p.pt[v] = fma(xd[v], kap, p.pt[v]);
#pragma unroll
    for (int i = 0; i < QL_SLOTS; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[i][0][v] = fma(x[i][v], kap, acc[i][0][v]);
    if (own && lk == 0) sh.rbuf[q * 16 + li] = li == q ? beta : fma(alpha - beta, kap, bc);  // row j of R
    if (wave == 0) {
      if (lk == 0) sh.zb[(li & 3) * 4 + (li >> 2)] = li < q ? ut * scal * p.scal : 0.0;  // v_c^T v_q
      ql_wave_sync();
      const ql_v4d z = reinterpret_cast<const ql_v4d*>(sh.zb)[lk];
      double ts = p.tr[0] * z[0];
#pragma unroll
      for (int i = 1; i <= HV; ++i) ts = fma(p.tr[i], z[i], ts);
      ts = -p.tau * ql_colsum(ts);
      ts = li == q ? p.tau : ts;
      if (lk == hk) p.tr[HV] = li <= q ? ts : 0.0;
    }
    p.scal = li == q ? scal : p.scal;
    p.beta = li == q ? beta : p.beta;
  }
}

// Factors panel P (held in acc): V and R back to A, T to Tt, |diag R| to D.
__device__ __attribute__((always_inline)) inline void ql_factor(QlBlock<1>& acc, const QrTask& tk, const QlShared& sh,
                                                                int P, ChainState* st) {
  const int N = tk.N, lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readlane((int)threadIdx.x >> 6, 0);
  const bool own = (P & (QL_WAVES - 1)) == wave;
  const int j0 = P << 4, w = min(16, N - j0);
  QlPanel p;
  p.scal = p.beta = p.tau = 0.0;
  p.zero = false;
  p.tr = ql_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    double e = 0.0;
#pragma unroll
    for (int i = 0; i < QL_SLOTS; ++i) {
      const double a = acc[i][0][v];
      e = QL_WAVES * i + wave == P ? a : e;
    }
    p.pt[v] = e;
  }
  ql_columns<0>(acc, p, sh, P, w);
  ql_columns<1>(acc, p, sh, P, w);
  ql_columns<2>(acc, p, sh, P, w);
  ql_columns<3>(acc, p, sh, P, w);
  LQMC_GLOBAL double* A = gptr(tk.A);
#pragma unroll
  for (int i = 0; i < QL_SLOTS; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int t = QL_WAVES * i + wave, r = 16 * t + lk + 4 * v;
      if (t > P && r < N && li < w) A[(size_t)r * N + j0 + li] = acc[i][0][v] * p.scal;
    }
  if (own) {
    ql_wave_sync();
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = lk + 4 * v;
      if (r < w && li < w) A[(size_t)(j0 + r) * N + j0 + li] = r > li ? p.pt[v] * p.scal : sh.rbuf[r * 16 + li];
    }
    if (lk == 0 && li < w) {
      const double d = fabs(p.beta);
      tk.D[j0 + li] = d > 0.0 ? d : 1e-300;
    }
    if (st && p.zero && lane == 0) atomicOr(&st[tk.chain].flags, 2u);
  }
  if (wave == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) tk.Tt[(size_t)P * 256 + li * 16 + lk + 4 * i] = p.tr[i];
  }
}

// Panel step P: block 0 of a matrix applies panel P - 1 to panel P and factors it, block k > 0
// applies panel P - 1 to the 32 columns from 16 (P + 1) + 32 (k - 1) on.
__global__ __launch_bounds__(QL_THREADS) void k_ql_step(const QrTask* __restrict__ tasks, int n, int nblk, int P,
                                                        ChainState* st) {
  // The factorising blocks of all matrices start first; a matrix's blocks, which read the same V,
  // have one residue mod 8 (one XCD).
  const int n8 = (n + 7) & ~7, b = blockIdx.x - n8, per = nblk - 1;
  const int k = b < 0 ? 0 : 1 + (b >> 3) % per;
  const int m = b < 0 ? (int)blockIdx.x : (b & 7) + 8 * ((b >> 3) / per);
  if (m >= n) return;
  const QrTask tk = tasks[m];
  const int N = tk.N;
  if (16 * P >= N) return;
  LQMC_DYNAMIC_LDS(double, sm);  // [8][2][64][4] partial products, tb, then QL_SHARED
  double* tb = sm + QL_WAVES * 2 * 256;
  if (k == 0) {
    QlShared sh;
    sh.xb = tb + QL_WAVES * QL_TB;
    sh.part = sh.xb + QL_WAVES * (QL_SLOTS + 1) * 16;
    sh.row = sh.part + 2 * QL_WAVES * 16;
    sh.rbuf = sh.row + 32;
    sh.zb = sh.rbuf + 256;
    QlBlock<1> acc;
    ql_load<1>(acc, tk, P > 0 ? P - 1 : 0, 16 * P);
    if (P > 0) {
      QlV p;
      ql_load_v<true>(p, tk, P - 1);
      ql_apply<1, true>(acc, p, tk, P - 1, -1, sm, tb);
      // row tile P - 1 of these columns is final
      const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
      const int wave = __builtin_amdgcn_readlane((int)threadIdx.x >> 6, 0);
#pragma unroll
      for (int i = 0; i < QL_SLOTS; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int t = QL_WAVES * i + wave, r = 16 * t + lk + 4 * v, c = 16 * P + li;
          if (t == P - 1 && c < N) gptr(tk.A)[(size_t)r * N + c] = acc[i][0][v];
        }
    }
    ql_factor(acc, tk, sh, P, st);
  } else {
    const int c0 = 16 * (P + 1) + 32 * (k - 1);
    if (P == 0 || c0 >= N) return;
    QlBlock<2> acc;
    QlV p;
    ql_load_v<true>(p, tk, P - 1);
    ql_load<2>(acc, tk, P - 1, c0);
    ql_apply<2, true>(acc, p, tk, P - 1, -1, sm, tb);
    ql_store<2>(acc, tk, P - 1, c0);
  }
}

// Q, 32 columns per workgroup: from the identity, the panels' reflectors from the last that reaches
// these columns to the first.
__global__ __launch_bounds__(QL_THREADS) void k_ql_formq(const QrTask* __restrict__ tasks, int nblk) {
  const int gb = xcd_grouped_block();
  const QrTask tk = tasks[gb / nblk];
  const int N = tk.N, c0 = 32 * (gb % nblk);
  if (c0 >= N) return;
  LQMC_DYNAMIC_LDS(double, sm);  // [8][2][64][4] partial products, tb
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readlane((int)threadIdx.x >> 6, 0);
  QlBlock<2> acc;
#pragma unroll
  for (int i = 0; i < QL_SLOTS; ++i)
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        acc[i][n][v] = 16 * (QL_WAVES * i + wave) + lk + 4 * v == c0 + 16 * n + li ? 1.0 : 0.0;
  int P = (min(N, c0 + 32) - 1) >> 4;
  QlV p;
  ql_load_v<false>(p, tk, P);
#pragma unroll 1
  for (; P >= 0; --P) ql_apply<2, false>(acc, p, tk, P, P - 1, sm, sm + QL_WAVES * 2 * 256);
#pragma unroll
  for (int i = 0; i < QL_SLOTS; ++i)
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int r = 16 * (QL_WAVES * i + wave) + lk + 4 * v, c = c0 + 16 * n + li;
        if (r < N && c < N) gptr(tk.Q)[(size_t)r * N + c] = acc[i][n][v];
      }
}

size_t ql_rows_shmem(int nmax) { return sizeof(double) * QL_ROWS * (size_t)nmax; }
size_t ql_order_shmem() { return sizeof(double) * QL_NMAX + sizeof(int) * 256; }
size_t ql_step_shmem() { return sizeof(double) * (QL_WAVES * (2 * 256 + QL_TB) + QL_SHARED); }
size_t ql_formq_shmem() { return sizeof(double) * QL_WAVES * (2 * 256 + QL_TB); }

int qr_large_limit() { return QL_NMAX; }

// QR with explicit Q of n matrices of at most nmax <= QL_NMAX.
void launch_qr_large(const QrTask* d, int n, int nmax, ChainState* st, hipStream_t s) {
  if (n <= 0) return;
  const int nb64 = (nmax + 63) / 64, nbr = (nmax + QL_ROWS - 1) / QL_ROWS, NS = (nmax + 15) / 16;
  hipLaunchKernelGGL(k_ql_norms, dim3(n * nb64), dim3(256), sizeof(double) * 256, s, d, nb64, st);
  hipLaunchKernelGGL(k_ql_order, dim3(n * nb64), dim3(256), ql_order_shmem(), s, d, nb64);
  hipLaunchKernelGGL(k_ql_gather, dim3(n * nbr), dim3(256), ql_rows_shmem(nmax), s, d, nbr);
  for (int P = 0; P < NS; ++P) {
    const int rest = nmax - 16 * (P + 1);
    const int nblk = 1 + (P > 0 && rest > 0 ? (rest + 31) / 32 : 0);
    hipLaunchKernelGGL(k_ql_step, dim3((n + 7) / 8 * 8 * nblk), dim3(QL_THREADS), ql_step_shmem(), s, d, n, nblk, P,
                       st);
  }
  hipLaunchKernelGGL(k_ql_out, dim3(n * nbr), dim3(256), ql_rows_shmem(nmax), s, d, nbr);
  const int nb32 = (nmax + 31) / 32;
  hipLaunchKernelGGL(k_ql_formq, dim3(n * nb32), dim3(QL_THREADS), ql_formq_shmem(), s, d, nb32);
}

}  // namespace lqmc
