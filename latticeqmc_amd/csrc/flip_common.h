// Device code shared by the flip kernels: the uniforms, and the end of a slice (exp(V) tables,
// counters and, on slice 0, the measurement).
#pragma once
#include "common.h"

#pragma clang fp contract(off)

namespace lqmc {

// ---- Philox4x32-10 (Salmon et al., SC'11) --------------------------------------------------
__device__ inline double philox_uniform(uint64_t seed, uint64_t q) {
  uint32_t c0 = (uint32_t)q, c1 = (uint32_t)(q >> 32), c2 = 0u, c3 = 0x51D3u;
  uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)(seed >> 32);
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint32_t lo0 = 0xD2511F53u * c0, hi0 = __umulhi(0xD2511F53u, c0);
    const uint32_t lo1 = 0xCD9E8D57u * c2, hi1 = __umulhi(0xCD9E8D57u, c2);
    const uint32_t n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
    c0 = n0; c1 = lo1; c2 = n2; c3 = lo0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  const double hi = (double)(c0 >> 5), lo = (double)(c1 >> 6);
  return (hi * 67108864.0 + lo) * (1.0 / 9007199254740992.0);
}

__device__ inline double draw_uniform(const ChainDev& ch, const ChainState* st, int chain, int rng,
                                      unsigned long long sweep, int t, int i, bool& underrun) {
  const unsigned long long NL = (unsigned long long)ch.N * ch.L;
  const unsigned long long within = (unsigned long long)t * ch.N + i;
  if (rng == 1) return philox_uniform(ch.seed, sweep * NL + within);
  const unsigned long long rel = sweep - st->replay_base;
  if (sweep < st->replay_base || rel >= st->replay_count) {
    underrun = true;
    return 2.0;  // rejects every ratio < 2; flagged
  }
  return ch.uni[rel * NL + within];
}

// ---- shared epilogue ---------------------------------------------------------------------------
__device__ inline double wg_sum(double v, double* red) {
  red[threadIdx.x] = v;
  __syncthreads();
  for (int s = blockDim.x >> 1; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  const double r = red[0];
  __syncthreads();
  return r;
}

// Measurement of one sweep from the equal-time G of both spins (lqmc.py:371-372 plus the
// per-sweep estimators): accumulate G, keep it as the last measured G, accumulate
// <S^z_i S^z_j>, and append density, double occupancy and kinetic energy per site to the
// chain's observable ring.  All threads of the workgroup take part (reductions).
template <typename T>
__device__ void measure_equal_time(const ChainDev& ch, ChainState* st, const T* G, double* red) {
  const int N = ch.N;
  {
    const size_t n2 = (size_t)N * N;
    for (size_t e = threadIdx.x; e < 2 * n2; e += blockDim.x) {
      const double g = (double)G[e];
      ch.Gacc[e] += g;
      ch.Glast[e] = g;
    }
    // <S^z_i S^z_j> by Wick's theorem for the sampled field, S^z = n_up - n_dn:
    // m_i m_j + sum_s (delta_ij - G_s,ji) G_s,ij with m_i = G_dn,ii - G_up,ii
    for (size_t e = threadIdx.x; e < n2; e += blockDim.x) {
      const size_t i = e / N, j = e % N;
      const double mi = (double)G[n2 + i * N + i] - (double)G[i * N + i];
      const double mj = (double)G[n2 + j * N + j] - (double)G[j * N + j];
      double v = mi * mj;
      for (int sp = 0; sp < 2; ++sp) {
        const double gij = (double)G[sp * n2 + i * N + j], gji = (double)G[sp * n2 + j * N + i];
        v += ((i == j ? 1.0 : 0.0) - gji) * gij;
      }
      ch.Sacc[e] += v;
    }
    double dens = 0.0, docc = 0.0, ek = 0.0;
    for (int i = threadIdx.x; i < N; i += blockDim.x) {
      const double nu = 1.0 - (double)G[(size_t)i * N + i];
      const double nd = 1.0 - (double)G[n2 + (size_t)i * N + i];
      dens += nu + nd;
      docc += nu * nd;
    }
    for (size_t e = threadIdx.x; e < n2; e += blockDim.x) {
      const size_t i = e / N, j = e % N;
      const double h = ch.hop[e];
      if (h != 0.0) ek -= h * ((double)G[j * N + i] + (double)G[n2 + j * N + i]);
    }
    dens = wg_sum(dens, red);
    docc = wg_sum(docc, red);
    ek = wg_sum(ek, red);
    if (threadIdx.x == 0) {
      const unsigned long long k = st->measured;
      double* o = ch.obs + (size_t)(k % (unsigned long long)ch.obs_cap) * 3;
      o[0] = dens / N;
      o[1] = docc / N;
      o[2] = ek / N;
      st->measured = k + 1;
    }
  }
}

template <typename T>
__device__ void slice_epilogue(const FlipArgs& a, const ChainDev& ch, int c, int l, const T* G,
                               unsigned long long nacc, bool underrun, bool bad, double* red) {
  const int N = ch.N;
  const int NL = N * ch.L;
  __syncthreads();
  for (int i = threadIdx.x; i < N; i += blockDim.x) {
    const int s = ch.field[(size_t)l * N + i];
    const double e1m = ch.e1m, e1p = ch.e1p;  // values, so the conditionals select values
    const double up = s > 0 ? e1m : e1p;
    const double dn = s > 0 ? e1p : e1m;
    ch.ev[(size_t)l * N + i] = up;
    ch.ev[(size_t)NL + (size_t)l * N + i] = dn;
    ch.evi[(size_t)l * N + i] = 1.0 / up;
    ch.evi[(size_t)NL + (size_t)l * N + i] = 1.0 / dn;
  }
  if (threadIdx.x == 0) {
    atomicAdd(&a.st[c].attempted, (unsigned long long)N);
    atomicAdd(&a.st[c].accepted, nacc);
    if (underrun) atomicOr(&a.st[c].flags, 4u);
    if (bad) atomicOr(&a.st[c].flags, 1u);
  }
  if (l == 0 && a.measure) measure_equal_time<T>(ch, &a.st[c], G, red);
  __syncthreads();
  if (l == 0 && threadIdx.x == 0) a.st[c].sweep += 1ull;
}

}  // namespace lqmc
