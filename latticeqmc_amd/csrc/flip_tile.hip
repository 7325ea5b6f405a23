// Metropolis flip phase of one time slice for chains whose Green's functions fit the registers of
// one workgroup (FP64, N <= 128).
//
// Both spins' G are loaded once, updated by Sherman-Morrison in registers for every accepted flip
// of the slice, and stored once.  Wavefronts 0 .. WR^2-1 hold spin up, the others spin down, each
// an 8T x 8T part of its spin; lane (a, b) = (l / 8, l % 8) holds rows a + 8 r and columns b + 8 j of
// the part, r, j < T.  Per site i (one workgroup barrier each):
//   the lanes that hold row i and column i of either spin put them into LDS (two buffers, by the
//   parity of i: a wavefront may be one site ahead of the slowest one);
//   after the barrier every wavefront reads both pivots G_ii, forms the ratio and the decision of
//   k_flip_rank1 (the same operations in the same order), reads its part of x = G[:, i] and
//   y = e_i - G[i, :], and on acceptance applies G -= x (c y)^T with T^2 multiply-adds.
// The results do not depend on T and WR.
//
// Bound by the latency of the site chain (LDS round trip, barrier, ratio, division) and, from about
// 64 sites on, by its T^2 multiply-adds; there are no block inverses, Z tiles or strip products, and
// G crosses the memory system once per slice.  Per launch, against the delayed kernel that these
// chains used before: 17.2 -> 8.2 us for one 4 x 4 chain, 69 -> 39 us for one 8 x 8 chain, 123 ->
// 65 us for 8 chains of 84 sites, 318 -> 95 us for 256 chains of 36, 64 and 100 sites, 169 -> 119 us
// for 32 chains of 117 sites.
#include "flip_common.h"

#include <algorithm>

#pragma clang fp contract(off)

namespace lqmc {

// num / d by Newton steps from the hardware reciprocal (d a determinant ratio, of order one).
__device__ inline double ft_div(double num, double d) {
#ifdef LQMC_CPU_EMU
  return num / d;
#else
  double r = __builtin_amdgcn_rcp(d);
  r = fma(fma(-d, r, 1.0), r, r);
  r = fma(fma(-d, r, 1.0), r, r);
  const double q = num * r;
  return fma(fma(-d, q, num), r, q);
#endif
}

template <int T, int WR>
__global__ __launch_bounds__(128 * WR * WR) void k_flip_tile(FlipArgs a) {
  constexpr int NP = 8 * T * WR;  // sites covered
  constexpr int PB = 4 * NP;      // one parity's buffers: rows of both spins, columns of both spins
  const int c = a.list ? a.list[blockIdx.x] : (int)blockIdx.x;
  const ChainDev ch = a.chains[c];
  if (a.t >= ch.L) return;
  const int N = ch.N;
  const int l = ch.L - 1 - a.t;
  const size_t n2 = (size_t)N * N;
  double* __restrict__ G = static_cast<double*>(ch.G);
  int8_t* fld = ch.field + (size_t)l * N;
  LQMC_DYNAMIC_LDS(double, sm);
  double* buf = sm;                // [2][PB]
  double* ub = buf + 2 * PB;       // [NP] uniforms
  double* e2 = ub + NP;            // [NP] exp(2 lambda s) of the slice's sites
  double* red = e2 + NP;           // blockDim (epilogue), and the trace of the slice before it
  int8_t* acc_sh = reinterpret_cast<int8_t*>(red + std::max((int)blockDim.x, NP));  // [NP] accepted
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readlane(tid >> 6, 0);
  const int sp = wave / (WR * WR), wr = (wave / WR) % WR, wc = wave % WR;
  const int la = lane >> 3, lb = lane & 7;
  const int r0 = 8 * T * wr + la, c0 = 8 * T * wc + lb;  // my first row and column
  bool underrun = false, bad = false;
  {
    const unsigned long long sweep = a.st[c].sweep;
    const double e2p = ch.e2p, e2m = ch.e2m;
    for (int i = tid; i < N; i += blockDim.x) {
      ub[i] = draw_uniform(ch, &a.st[c], c, a.rng, sweep, a.t, i, underrun);
      e2[i] = fld[i] > 0 ? e2p : e2m;
    }
  }
  double g[T][T];
  {
    const LQMC_GLOBAL double* Gs = gptr(G) + sp * n2;
#pragma unroll
    for (int r = 0; r < T; ++r)
#pragma unroll
      for (int j = 0; j < T; ++j) {
        const int row = r0 + 8 * r, col = c0 + 8 * j;
        g[r][j] = ldg0(Gs, (size_t)row * N + col, row < N && col < N);
      }
  }
  unsigned long long nacc = 0;
#pragma unroll 1
  for (int q = 0; q < WR; ++q) {
#pragma unroll
    for (int k = 0; k < T; ++k) {
#pragma unroll 1
      for (int o = 0; o < 8; ++o) {
        const int i = 8 * (T * q + k) + o;
        if (i >= N) break;
        double* pb = buf + (i & 1) * PB;
        double* rowb = pb + sp * NP;           // row i of my spin
        double* colb = pb + (2 + sp) * NP;     // column i of my spin
        if (wr == q && la == o) {
#pragma unroll
          for (int j = 0; j < T; ++j) rowb[c0 + 8 * j] = g[k][j];
        }
        if (wc == q && lb == o) {
#pragma unroll
          for (int r = 0; r < T; ++r) colb[r0 + 8 * r] = g[r][k];
        }
        __syncthreads();
        const double gu = pb[i], gd = pb[NP + i], u = ub[i], ep = e2[i];
        double x[T], y[T];
#pragma unroll
        for (int r = 0; r < T; ++r) x[r] = colb[r0 + 8 * r];
#pragma unroll
        for (int j = 0; j < T; ++j) y[j] = rowb[c0 + 8 * j];
        const double em = ep == ch.e2p ? ch.e2m : ch.e2p;
        const double d_up = 1.0 + (1.0 - gu) * (ep - 1.0);
        const double d_dn = 1.0 + (1.0 - gd) * (em - 1.0);
        const double ratio = d_up * d_dn;
        const bool acc = u <= ratio;
        if (!isfinite(ratio)) bad = true;
        if (tid == 0) {
          acc_sh[i] = acc ? 1 : 0;
          if (a.trace) red[i] = ratio;
        }
        if (acc) {
          ++nacc;
          // y = e_i - G[i, :], coefficient alpha / (1 + alpha (1 - G_ii)) of my spin
          const double cf = sp == 0 ? ft_div(ep - 1.0, d_up) : ft_div(em - 1.0, d_dn);
          double cy[T];
#pragma unroll
          for (int j = 0; j < T; ++j) {
            const double yj = c0 + 8 * j == i ? 1.0 - y[j] : -y[j];
            cy[j] = cf * yj;
          }
#pragma unroll
          for (int r = 0; r < T; ++r)
#pragma unroll
            for (int j = 0; j < T; ++j) g[r][j] = fma(-cy[j], x[r], g[r][j]);
        }
      }
    }
  }
  {
    LQMC_GLOBAL double* Gs = gptr(G) + sp * n2;
#pragma unroll
    for (int r = 0; r < T; ++r)
#pragma unroll
      for (int j = 0; j < T; ++j) {
        const int row = r0 + 8 * r, col = c0 + 8 * j;
        if (row < N && col < N) Gs[(size_t)row * N + col] = g[r][j];
      }
  }
  __syncthreads();
  for (int i = tid; i < N; i += blockDim.x) {
    if (a.trace) {
      ch.tr_ratio[(size_t)a.t * N + i] = red[i];
      ch.tr_acc[(size_t)a.t * N + i] = (uint8_t)acc_sh[i];
    }
    if (acc_sh[i]) fld[i] = (int8_t)(-fld[i]);
  }
  slice_epilogue<double>(a, ch, c, l, G, nacc, underrun, bad, red);
}

// Sites covered by class k of the kernel's forms (rising; the last one is the limit of its use).
static const int kTileSites[] = {16, 32, 48, 64, 80, 96, 112, 128};
int flip_tile_limit() { return 128; }
// The smallest form that covers N sites, or -1.
int flip_tile_class(int N) {
  for (int k = 0; k < 8; ++k)
    if (N <= kTileSites[k]) return k;
  return -1;
}

template <int T, int WR>
static void ft_launch(const FlipArgs& a, hipStream_t s) {
  constexpr int threads = 128 * WR * WR, NP = 8 * T * WR;
  const size_t sh = sizeof(double) * (8 * NP + 2 * NP + std::max(threads, NP)) + NP;
  hipLaunchKernelGGL((k_flip_tile<T, WR>), dim3(a.nchains), dim3(threads), sh, s, a);
}

// The flips of a.nchains chains (a.list) of at most kTileSites[cls] sites.  Up to 32 sites two
// wavefronts hold a chain (a barrier between two of them is the cheapest), above that eight.
void launch_flip_tile(int cls, const FlipArgs& a, hipStream_t s) {
  if (a.nchains <= 0) return;
  switch (cls) {
    case 0: ft_launch<2, 1>(a, s); break;
    case 1: ft_launch<4, 1>(a, s); break;
    case 2: ft_launch<3, 2>(a, s); break;
    case 3: ft_launch<4, 2>(a, s); break;
    case 4: ft_launch<5, 2>(a, s); break;
    case 5: ft_launch<6, 2>(a, s); break;
    case 6: ft_launch<7, 2>(a, s); break;
    default: ft_launch<8, 2>(a, s); break;
  }
}

}  // namespace lqmc
