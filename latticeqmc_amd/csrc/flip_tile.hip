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

// Both spins' matrices of the wrap in LDS at once (up to 96 sites), or one after the other.
constexpr int ft_wrap_spins(int NP) { return NP <= 96 ? 2 : 1; }

typedef double ft_v4d __attribute__((ext_vector_type(4)));

__device__ inline ft_v4d ft_mma(double a, double b, ft_v4d c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }

// The matrix-core A operands of the wrap's four directions: Eyi, Exi (by rows), Ey, Ex (by columns).
struct FtWrapE { double e[4][4]; };
__device__ inline void ft_wrap_load(FtWrapE& w, const LQMC_GLOBAL double* kr, int lane) {
  const int li = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int kk = 4 * s + lk;
    w.e[0][s] = kr[768 + li * 16 + kk];
    w.e[1][s] = kr[512 + li * 16 + kk];
    w.e[2][s] = kr[256 + kk * 16 + li];
    w.e[3][s] = kr[kk * 16 + li];
  }
}

// Fibers of n entries, st apart, in LDS: fiber f = (o, i), i < N, of total starts at o so + i sf, o from count
// on belonging to the second matrix, V2 further on.  Each is multiplied by the n x n matrix of the operands e,
// in place, 16 fibers per wavefront and product, Q products in flight, KS = ceil(n / 4).  The latency of a
// wavefront's own instructions is what these small products cost, so the loop is kept free of predicates: lanes
// past the last fiber repeat it (and do not write), entries past n are read from the zero at V[zero].
template <int WAVES, int KS, int Q>
__device__ __attribute__((always_inline)) inline void ft_wrap_stage(double* V, const double (&e)[4], int n, int st, int N,
                                                                    unsigned magic, int count, int total, int so, int sf,
                                                                    int V2, int zero, int wave, int lane) {
  const int li = lane & 15, lk = lane >> 4;
  constexpr int HOP = 16 * WAVES;
  const bool last = lk + 4 * (KS - 1) < n;  // my last entry is inside the fiber
  const int os = so - N * sf, v2 = V2 - count * so, l0 = lk * st;
#pragma unroll 1
  for (int f0 = 16 * wave; f0 < total; f0 += Q * HOP) {
    int v[Q];  // my first entry of my fiber
    double b[Q][KS];
    ft_v4d acc[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      // (a product past the last fiber repeats the first one of its step and is not written)
      const int f = std::min(f0 + (f0 + q * HOP < total ? q * HOP : 0) + li, total - 1);
      const int o = (int)__umulhi((unsigned)f, magic);
      v[q] = f * sf + o * os + (o >= count ? v2 : 0) + l0;
#pragma unroll
      for (int s = 0; s < KS; ++s) b[q][s] = V[s < KS - 1 || last ? v[q] + 4 * s * st : zero];
      acc[q] = ft_v4d{0.0, 0.0, 0.0, 0.0};
    }
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int q = 0; q < Q; ++q) acc[q] = ft_mma(e[s], b[q][s], acc[q]);
#pragma unroll
    for (int q = 0; q < Q; ++q)
      if (f0 + q * HOP + li < total) {
#pragma unroll
        for (int r = 0; r < KS - 1; ++r) V[v[q] + 4 * r * st] = acc[q][r];
        if (last) V[v[q] + 4 * (KS - 1) * st] = acc[q][KS - 1];
      }
  }
}

// V <- (Exi (x) Eyi) V (Ex (x) Ey) for the ns N x N matrices V (row stride ld, V2 apart) in LDS, one direction
// of one side at a time, a barrier after each; V[ns V2] is zero.
template <int WAVES, int Q4>
__device__ __attribute__((always_inline)) inline void ft_wrap_products(double* V, const FtWrapE& w, int ns, int N, int ld, int V2,
                                                                       int n1, int n2, int wave, int lane) {
  // f / N = umulhi(f, magic): exact while f N < 2^32, f < 2 * 128 * 16
  const unsigned magic = 0xFFFFFFFFu / (unsigned)N + 1u;
#pragma unroll
  for (int stage = 0; stage < 4; ++stage) {
    const bool right = stage >= 2, x = stage & 1;
    const int n = x ? n1 : n2, count = x ? n2 : n1;
    const int st = right ? (x ? n2 : 1) : (x ? n2 * ld : ld);
    const int so = (right ? 1 : ld) * (x ? 1 : n2), sf = right ? ld : 1;
#define FT_STAGE(KS, Q) \
  ft_wrap_stage<WAVES, KS, Q>(V, w.e[stage], n, st, N, magic, count, ns * N * count, so, sf, V2, ns * V2, wave, lane)
    switch ((n + 3) >> 2) {
      case 1: FT_STAGE(1, Q4); break;
      case 2: FT_STAGE(2, Q4); break;
      case 3: FT_STAGE(3, 2); break;
      default: FT_STAGE(4, 2); break;
    }
#undef FT_STAGE
    __syncthreads();
  }
}

// A chain's description, read anew: held over the slices of a launch it would fill the registers.
__device__ inline ChainDev ft_chain(const ChainDev* p) {
  const LQMC_CONST ChainDev* q = uniform_const(p);
  LQMC_OPAQUE(q, "s");
  ChainDev ch;
  __builtin_memcpy(&ch, (const ChainDev*)q, sizeof ch);
  return ch;
}

// WRAP (chains with a factored E_K): the wrap G <- E_K^-1 V^-1 G V E_K of the slice follows in the same
// launch, through LDS, and the launch runs a.slices slices, G staying in registers between them.
template <int T, int WR, bool WRAP = false>
__global__ __launch_bounds__(128 * WR * WR) void k_flip_tile(FlipArgs a) {
  constexpr int NP = 8 * T * WR;  // sites covered
  constexpr int PB = 4 * NP;      // one parity's buffers: rows of both spins, columns of both spins
  const int c = a.list ? a.list[blockIdx.x] : (int)blockIdx.x;
  const ChainDev ch = a.chains[c];
  if (a.t >= ch.L) return;
  const int N = ch.N;
  const size_t n2 = (size_t)N * N;
  double* __restrict__ G = static_cast<double*>(ch.G);
  LQMC_DYNAMIC_LDS(double, sm);
  double* buf = sm;                // [2][PB]
  double* ub = buf + 2 * PB;       // [NP] uniforms
  double* red = ub + NP;           // blockDim (epilogue), and the slice's ratios before it (trace)
  int* neg_sh = reinterpret_cast<int*>(red + std::max((int)blockDim.x, NP));  // [NP] spin is -1
  int* acc_sh = neg_sh + NP;       // [NP / 8] accepted, a bit per site
  double* const vw = reinterpret_cast<double*>(acc_sh + NP / 8);  // WRAP: [ft_wrap_spins(NP)][NP][NP + 1], a zero
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readlane(tid >> 6, 0);
  const int sp = wave / (WR * WR), wr = (wave / WR) % WR, wc = wave % WR;
  const int la = lane >> 3, lb = lane & 7;
  const int r0 = 8 * T * wr + la, c0 = 8 * T * wc + lb;  // my first row and column
  bool underrun = false;
  const unsigned long long sweep = a.st[c].sweep;
  double un = 2.0;  // uniform and sign of site tid in the coming slice
  int nn = 0;
  auto draw = [&](int t) {
    const ChainDev ch = ft_chain(a.chains + c);
    if (tid < N) {
      nn = ch.field[(size_t)(ch.L - 1 - t) * N + tid] < 0 ? 1 : 0;
      un = draw_uniform(ch, &a.st[c], c, a.rng, sweep, t, tid, underrun);
    }
  };
  draw(a.t);
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
  auto store = [&] {
    LQMC_GLOBAL double* Gs = gptr(G) + sp * n2;
#pragma unroll
    for (int r = 0; r < T; ++r)
#pragma unroll
      for (int j = 0; j < T; ++j) {
        const int row = r0 + 8 * r, col = c0 + 8 * j;
        if (row < N && col < N) Gs[(size_t)row * N + col] = g[r][j];
      }
  };
  const double ap = ch.e2p - 1.0, am = ch.e2m - 1.0;  // alpha of a spin +1 (sigma = +1), and of a spin -1
  double* const rowb = buf + sp * NP + c0;            // my part of row i of my spin
  double* const colb = buf + (2 + sp) * NP + r0;      // my part of column i of my spin
  FtWrapE we;
  if constexpr (WRAP && T < 6) ft_wrap_load(we, gptr(ch.kr), lane);
  // WRAP: V of a spin +1 and -1 and their inverses, as in the exp(V) tables
  double ep = sp == 0 ? ch.e1m : ch.e1p, en = sp == 0 ? ch.e1p : ch.e1m;
  double epi = 1.0 / ep, eni = 1.0 / en;
  if constexpr (WRAP) {
    LQMC_OPAQUE(epi, "v");
    LQMC_OPAQUE(eni, "v");
    if (tid == 0) vw[ft_wrap_spins(NP) * NP * (NP + 1)] = 0.0;
  }
  const int tend = WRAP ? std::min(a.t + a.slices, ch.L) : a.t + 1;
#pragma unroll 1
  for (int t = a.t; t < tend; ++t) {
    const int l = ch.L - 1 - t;
    unsigned nacc = 0;
    double fin = 0.0;  // becomes NaN with the first ratio that is not finite
    if (tid < NP) {
      ub[tid] = un;
      neg_sh[tid] = nn;
    }
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
    if (!WRAP || (l == 0 && a.measure)) store();
    const ChainDev ce = ft_chain(a.chains + c);
    if (WRAP && t + 1 < tend) draw(t + 1);
    __syncthreads();
    if (tid < N) {
      const int acc = (acc_sh[tid >> 3] >> (tid & 7)) & 1;
      if (a.trace) {
        ce.tr_ratio[(size_t)t * N + tid] = red[tid];
        ce.tr_acc[(size_t)t * N + tid] = (uint8_t)acc;
      }
      if (acc) {
        ce.field[(size_t)l * N + tid] = (int8_t)(neg_sh[tid] ? 1 : -1);
        if (WRAP) neg_sh[tid] ^= 1;
      }
    }
    // the wrap's operands and addresses are formed anew: kept across the slices they would fill the registers
    int ln = lane;
    LQMC_OPAQUE(ln, "v");
    if constexpr (WRAP && T >= 6) ft_wrap_load(we, gptr(ce.kr), ln);
    slice_epilogue<double>(a, ce, c, l, G, nacc, underrun, !(fin == 0.0), red);
    if constexpr (WRAP) {
      constexpr int NS = ft_wrap_spins(NP), ld = NP + 1;
      double* const mine = vw + (NS == 2 ? sp : 0) * NP * ld + r0 * ld + c0;
#pragma unroll 1
      for (int pass = 0; pass < 2 / NS; ++pass) {
        const bool my = NS == 2 || pass == sp;
        if (my) {
          double vc[T];
#pragma unroll
          for (int j = 0; j < T; ++j) vc[j] = neg_sh[c0 + 8 * j] ? en : ep;
#pragma unroll
          for (int r = 0; r < T; ++r) {
            const double vr = neg_sh[r0 + 8 * r] ? eni : epi;
#pragma unroll
            for (int j = 0; j < T; ++j)
              mine[8 * r * ld + 8 * j] = vr * g[r][j] * vc[j];  // zero past the last site
          }
        }
        __syncthreads();
        ft_wrap_products<2 * WR * WR, (T < 6 ? 4 : 2)>(vw, we, NS, N, ld, NP * ld, ce.kn1, ce.kn2, wave, ln);
        if (my) {
#pragma unroll
          for (int r = 0; r < T; ++r)
#pragma unroll
            for (int j = 0; j < T; ++j)
              g[r][j] = mine[8 * r * ld + 8 * j];
        }
        if (NS == 1) __syncthreads();
      }
    }
  }
  if (WRAP) store();
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
constexpr size_t ft_shmem(bool wrap) {
  constexpr int threads = 128 * WR * WR, NP = 8 * T * WR;
  return sizeof(double) * (9 * NP + std::max(threads, NP)) + sizeof(int) * (NP + NP / 8) +
         (wrap ? sizeof(double) * (ft_wrap_spins(NP) * NP * (NP + 1) + 1) : 0);
}

template <int T, int WR>
static void ft_launch(const FlipArgs& a, hipStream_t s) {
  constexpr int threads = 128 * WR * WR;
  if (a.slices > 0) hipLaunchKernelGGL((k_flip_tile<T, WR, true>), dim3(a.nchains), dim3(threads), (ft_shmem<T, WR>(true)), s, a);
  else hipLaunchKernelGGL((k_flip_tile<T, WR>), dim3(a.nchains), dim3(threads), (ft_shmem<T, WR>(false)), s, a);
}

// LDS of class cls with the wraps.
size_t flip_tile_wrap_shmem(int cls) {
  switch (cls) {
    case 0: return ft_shmem<2, 1>(true);
    case 1: return ft_shmem<4, 1>(true);
    case 2: return ft_shmem<3, 2>(true);
    case 3: return ft_shmem<4, 2>(true);
    case 4: return ft_shmem<5, 2>(true);
    case 5: return ft_shmem<6, 2>(true);
    case 6: return ft_shmem<7, 2>(true);
    default: return ft_shmem<8, 2>(true);
  }
}

// The flips of a.nchains chains (a.list) of at most kTileSites[cls] sites, with the wraps of a.slices
// slices when that is set (chains with kn1 > 0 only).  Up to 32 sites two
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
