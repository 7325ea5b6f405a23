// One lattice direction of a Kronecker-factored product, in place, on the vector units: a thread
// holds a fiber v[0], v[st], ... (n entries of the contracted direction) in registers and writes
// E v over it.  The rows of E come through scalar loads (they are the same for every thread), so a
// step is one multiply-add per entry with no operand traffic; FP64 matrix instructions have the
// same peak rate and pad every direction to 16.
#pragma once
#include "common.h"

namespace lqmc {

// v[b st] <- sum_k E[b ld + k] v[k st], b, k < n; n is F or F - 1 (E is zero past n up to row and column F).
template <int F>
__device__ __attribute__((always_inline)) inline void kf_fiber(double* v, int st, const LQMC_CONST double* E, int ld, int n) {
  double in[F];
#pragma unroll
  for (int k = 0; k < F - 1; ++k) in[k] = v[k * st];
  in[F - 1] = n == F ? v[(F - 1) * st] : 0.0;
  if constexpr (F <= 16) {
#pragma unroll 1
    for (int b = 0; b < n; b += 2) {
      const LQMC_CONST double* e0 = E + b * ld;
      const LQMC_CONST double* e1 = e0 + ld;
      double s0 = 0.0, s1 = 0.0;
#pragma unroll
      for (int k = 0; k < F; ++k) {
        s0 = fma(e0[k], in[k], s0);
        s1 = fma(e1[k], in[k], s1);
      }
      v[b * st] = s0;
      if (b + 1 < n) v[(b + 1) * st] = s1;
    }
  } else {  // one row: two of them would not fit the scalar registers
#pragma unroll 1
    for (int b = 0; b < n; ++b) {
      const LQMC_CONST double* e0 = E + b * ld;
      double s0 = 0.0;
#pragma unroll
      for (int k = 0; k < F; ++k) s0 = fma(e0[k], in[k], s0);
      v[b * st] = s0;
    }
  }
}

// kf_fiber for n in 2 .. LIMIT (uniform), LIMIT 16 or 32.
template <int LIMIT>
__device__ __attribute__((always_inline)) inline void kf_apply(double* v, int st, const LQMC_CONST double* E, int ld, int n) {
  switch ((n + 1) >> 1) {
    case 1: kf_fiber<2>(v, st, E, ld, n); break;
    case 2: kf_fiber<4>(v, st, E, ld, n); break;
    case 3: kf_fiber<6>(v, st, E, ld, n); break;
    case 4: kf_fiber<8>(v, st, E, ld, n); break;
    case 5: kf_fiber<10>(v, st, E, ld, n); break;
    case 6: kf_fiber<12>(v, st, E, ld, n); break;
    case 7: kf_fiber<14>(v, st, E, ld, n); break;
    case 8: kf_fiber<16>(v, st, E, ld, n); break;
    default:
      if constexpr (LIMIT > 16) {
        switch ((n + 1) >> 1) {
          case 9: kf_fiber<18>(v, st, E, ld, n); break;
          case 10: kf_fiber<20>(v, st, E, ld, n); break;
          case 11: kf_fiber<22>(v, st, E, ld, n); break;
          case 12: kf_fiber<24>(v, st, E, ld, n); break;
          case 13: kf_fiber<26>(v, st, E, ld, n); break;
          case 14: kf_fiber<28>(v, st, E, ld, n); break;
          case 15: kf_fiber<30>(v, st, E, ld, n); break;
          default: kf_fiber<32>(v, st, E, ld, n); break;
        }
      }
  }
}

}  // namespace lqmc
