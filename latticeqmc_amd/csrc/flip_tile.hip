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
// Bound by the latency of the site chain (LDS round trip, barrier, ratio, division: about 900 cycles,
// whatever T) and, from about 100 sites on, by the issue of its T^2 multiply-adds; there are no
// block inverses, Z tiles or strip products, and G crosses the memory system once per slice.  The
// uniforms and signs of eight sites are picked from registers, the parity of the buffers is a
// constant and y's unit entry touches one register, which took a fifth off the chain.  Per launch,
// against the delayed kernel that these chains used before: 17.2 -> 7.6 us for one 4 x 4 chain,
// 69 -> 33 us for one 8 x 8 chain, 318 -> 82 us for 256 chains of 36, 64 and 100 sites.
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

// Lane l's value (l wavefront-uniform) in scalar registers.
__device__ inline double ft_readlane(double v, int l) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
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
  double* red = ub + NP;           // blockDim (epilogue), and the slice's ratios before it (trace)
  int* neg_sh = reinterpret_cast<int*>(red + std::max((int)blockDim.x, NP));  // [NP] spin is -1
  int* acc_sh = neg_sh + NP;       // [NP / 8] accepted, a bit per site
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readlane(tid >> 6, 0);
  const int sp = wave / (WR * WR), wr = (wave / WR) % WR, wc = wave % WR;
  const int la = lane >> 3, lb = lane & 7;
  const int r0 = 8 * T * wr + la, c0 = 8 * T * wc + lb;  // my first row and column
  bool underrun = false;
  {
    const unsigned long long sweep = a.st[c].sweep;
    for (int i = tid; i < NP; i += blockDim.x) {
      ub[i] = i < N ? draw_uniform(ch, &a.st[c], c, a.rng, sweep, a.t, i, underrun) : 2.0;
      neg_sh[i] = i < N && fld[i] < 0 ? 1 : 0;
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
  const double ap = ch.e2p - 1.0, am = ch.e2m - 1.0;  // alpha of a spin +1 (sigma = +1), and of a spin -1
  double* const rowb = buf + sp * NP + c0;            // my part of row i of my spin
  double* const colb = buf + (2 + sp) * NP + r0;      // my part of column i of my spin
  unsigned nacc = 0;
  double fin = 0.0;  // becomes NaN with the first ratio that is not finite
  __syncthreads();
#pragma unroll 1
  for (int q = 0; q < WR; ++q) {
#pragma unroll
    for (int k = 0; k < T; ++k) {
      const int i0 = 8 * (T * q + k);
      if (i0 >= N) break;
      // the uniforms and signs of these eight sites, site o in the lanes with lb = o
      const double ul = ub[i0 + lb];
      const int nl = neg_sh[i0 + lb];
      unsigned abits = 0;
#pragma unroll 1
      for (int o2 = 0; o2 < 8; o2 += 2) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {  // the buffers' parity
          const int o = o2 + h, i = i0 + o;
          if (i >= N) break;
          if (wr == q && la == o) {
#pragma unroll
            for (int j = 0; j < T; ++j) rowb[h * PB + 8 * j] = g[k][j];
          }
          if (wc == q && lb == o) {
#pragma unroll
            for (int r = 0; r < T; ++r) colb[h * PB + 8 * r] = g[r][k];
          }
          const double u = ft_readlane(ul, o);
          const bool neg = __builtin_amdgcn_readlane(nl, o) != 0;
          const double al_up = neg ? am : ap, al_dn = neg ? ap : am;
          __syncthreads();
          const double gu = buf[h * PB + i], gd = buf[h * PB + NP + i];
          double x[T], y[T];
#pragma unroll
          for (int r = 0; r < T; ++r) x[r] = colb[h * PB + 8 * r];
#pragma unroll
          for (int j = 0; j < T; ++j) y[j] = rowb[h * PB + 8 * j];
          const double d_up = 1.0 + (1.0 - gu) * al_up;
          const double d_dn = 1.0 + (1.0 - gd) * al_dn;
          const double ratio = d_up * d_dn;
          if (a.trace && tid == 0) red[i] = ratio;
          fin = fma(ratio, 0.0, fin);
          if (u <= ratio) {
            ++nacc;
            abits |= 1u << o;
            // G -= x (cf y)^T, y = e_i - G[i, :], cf = alpha / (1 + alpha (1 - G_ii)) of my spin
            const double cf = ft_div(sp == 0 ? al_up : al_dn, sp == 0 ? d_up : d_dn);
            if (wc == q && lb == o) y[k] -= 1.0;
#pragma unroll
            for (int j = 0; j < T; ++j) y[j] = cf * y[j];
#pragma unroll
            for (int r = 0; r < T; ++r)
#pragma unroll
              for (int j = 0; j < T; ++j) g[r][j] = fma(y[j], x[r], g[r][j]);
          }
        }
      }
      if (tid == 0) acc_sh[i0 >> 3] = (int)abits;
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
    const int acc = (acc_sh[i >> 3] >> (i & 7)) & 1;
    if (a.trace) {
      ch.tr_ratio[(size_t)a.t * N + i] = red[i];
      ch.tr_acc[(size_t)a.t * N + i] = (uint8_t)acc;
    }
    if (acc) fld[i] = (int8_t)(neg_sh[i] ? 1 : -1);
  }
  slice_epilogue<double>(a, ch, c, l, G, nacc, underrun, !(fin == 0.0), red);
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
  const size_t sh = sizeof(double) * (9 * NP + std::max(threads, NP)) + sizeof(int) * (NP + NP / 8);
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
