// Products with the kinetic propagator E_K = exp(-dtau K) of a lattice whose hopping matrix is a
// Kronecker sum, K = Kx (x) I + I (x) Ky (the square and cubic lattices with uniform hopping per
// direction).  Then E_K = Ex (x) Ey exactly, and with the site index i = a n2 + b a column x of
// the operand, read as the n1 x n2 array M[a][b] = x[a n2 + b], maps to Ex M Ey^T.  A product
// E X (N x N, N = n1 n2) costs 2 N^2 (n1 + n2) flops instead of 2 N^3, and each launch reads
// and writes its operands once: at N = 256 a memory-bound pass in place of a 256^3 GEMM.
//
// One 256-thread workgroup per 16 columns of X (left product E X) or 16 rows of X (right
// product X E, handled as E^T X^T).  The tile goes to LDS as V[a'][b'][j] (the k index split
// into its two lattice coordinates), the four wavefronts contract b' with Ey on the matrix
// cores (16x16x4 FP64, one 16 x 16 x 16 product per a'), then a' with Ex (one per b), and
// write the result with the diagonal scales of the task applied.
#include "common.h"
#include "kron_fiber.h"

#include <algorithm>

namespace lqmc {

typedef double kr_v4d __attribute__((ext_vector_type(4)));

constexpr int KR_T = 16;             // columns (left) or rows (right) of X per workgroup
constexpr int KR_BS = 17;            // LDS stride of b' (odd: transposed writes spread over banks)
constexpr int KR_AS = 16 * KR_BS;    // LDS stride of a'

__device__ inline kr_v4d kr_mma(double a, double b, kr_v4d c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Index of the task holding tile `tile` (tasks sorted by tile_base).
template <typename Task>
__device__ inline int kr_task(const Task* __restrict__ tasks, int ntasks, int tile) {
  int lo = 0, hi = ntasks - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (tasks[mid].tile_base <= tile) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Element u of this thread's share of tile `tile`'s operand: V[a'][b'][j] with e = tid + 256 u,
// the fastest index of e running along memory (j for the left product, b' for the right one).
template <bool RIGHT>
__device__ inline void kr_coords(int e, int& ap, int& bp, int& j) {
  j = RIGHT ? e >> 8 : e & 15;
  bp = RIGHT ? e & 15 : (e >> 4) & 15;
  ap = RIGHT ? (e >> 4) & 15 : e >> 8;
}

// A diagonal scale entry from its stored value (the kinds of scale_val).
__device__ inline double kr_scale_of(int kind, double v) {
  switch (kind) {
    case SC_PLAIN: return v;
    case SC_INV: return 1.0 / v;
    case SC_INV_BIG: return 1.0 / fmax(v, 1.0);
    case SC_SMALL: return fmin(v, 1.0);
    default: return 1.0;
  }
}

// The tile's operand share (v) and entry tid of the task's three scale vectors (raw).
template <bool RIGHT, bool F16>
__device__ inline void kr_load(const KronTask& tk, int t0, double (&v)[16], double (&sc)[3]) {
  const int tid = threadIdx.x;
  sc[0] = tk.ks_kind != SC_NONE && tid < tk.N ? tk.ks[tid] : 1.0;
  sc[1] = tk.rs_kind != SC_NONE && tid < tk.N ? tk.rs[tid] : 1.0;
  sc[2] = tk.cs_kind != SC_NONE && tid < tk.N ? tk.cs[tid] : 1.0;
  const LQMC_GLOBAL double* X = gptr(tk.X);
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    int ap, bp, j;
    kr_coords<RIGHT>((int)threadIdx.x + 256 * u, ap, bp, j);
    const bool ok = F16 || (ap < tk.n1 && bp < tk.n2 && t0 + j < tk.N);
    const int k = ap * tk.n2 + bp;
    const size_t ix = RIGHT ? (size_t)(t0 + j) * tk.ldx + k : (size_t)k * tk.ldx + t0 + j;
    if constexpr (F16) v[u] = X[ix];
    else v[u] = ldg0(X, ix, ok);
  }
}

// RIGHT: C = diag(rs) X diag(ks) E diag(cs), computed as the left product with E^T = Ex^T (x) Ey^T
// applied to the rows of X.  Each workgroup walks tiles blockIdx.x, + gridDim.x, ...; the next
// tile's operand loads are issued before the current tile's contractions, so they are in flight
// during them.
template <bool RIGHT, bool F16>
__global__ __launch_bounds__(256, 4) void k_kron(const KronTask* __restrict__ tasks, int ntasks, int ntiles) {
  int tile = blockIdx.x;
  if (tile >= ntiles) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lk = lane >> 4;
  LQMC_DYNAMIC_LDS(double, vs);  // [16 a'][16 b' (stride KR_BS)][16 j], then ks, rs, cs [256] each
  double* const ksl = vs + 16 * KR_AS;
  double* const rsl = ksl + 256;
  double* const csl = rsl + 256;
  KronTask tk = tasks[kr_task(tasks, ntasks, tile)];
  int t0 = (tile - tk.tile_base) * KR_T;  // first column (left) or row (right) of the tile
  double v[16], sc[3];
  kr_load<RIGHT, F16>(tk, t0, v, sc);
  for (;;) {
    // F16: every task of the launch is 16 x 16 (N = 256): no tile reaches past the lattice
    const int N = F16 ? 256 : tk.N, n1 = F16 ? 16 : tk.n1, n2 = F16 ? 16 : tk.n2;
    // 1. V[a'][b'][j] = X[k][t0 + j] (left) or X[t0 + j][k] (right), k = a' n2 + b'; zero outside
    //    a' < n1, b' < n2, t0 + j < N.  The scales to LDS (ks is applied to the stage-1 operands).
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      int ap, bp, j;
      kr_coords<RIGHT>(tid + 256 * u, ap, bp, j);
      vs[ap * KR_AS + bp * KR_BS + j] = v[u];
    }
    ksl[tid] = kr_scale_of(tk.ks_kind, sc[0]);
    rsl[tid] = kr_scale_of(tk.rs_kind, sc[1]);
    csl[tid] = kr_scale_of(tk.cs_kind, sc[2]);
    // the A operands: lane holds F[row li][k 4s + lk] of F = Ey (stage 1) and Ex (stage 2), or
    // their transposes for the right product; zero past n2 / n1
    double ay[4], ax[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int kk = 4 * s + lk;
      ay[s] = tk.Ey[RIGHT ? kk * 16 + li : li * 16 + kk];
      ax[s] = tk.Ex[RIGHT ? kk * 16 + li : li * 16 + kk];
    }
    // the next tile's operand, in flight during the contractions below
    const int nt = tile + (int)gridDim.x;
    const bool more = nt < ntiles;
    KronTask tn = tk;
    int n0 = 0;
    if (more) {
      tn = tasks[kr_task(tasks, ntasks, nt)];
      n0 = (nt - tn.tile_base) * KR_T;
      kr_load<RIGHT, F16>(tn, n0, v, sc);
    }
    __syncthreads();

    // 2. T[a'][b][j] = sum_b' Ey[b][b'] ks[k] V[a'][b'][j] for this wavefront's a' = wave + 8h + 4q
    //    (in place: each a' block is read and written by one wavefront only; blocks past n1
    //    hold zeros and stay zero)
    // two a' blocks at a time (register budget of four workgroups per compute unit)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      kr_v4d acc[2];
      double bv[2][4];
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int ap = wave + 8 * h + 4 * q, bp = 4 * s + lk;
          const double kf = F16 || (ap < n1 && bp < n2) ? ksl[ap * n2 + bp] : 0.0;
          bv[q][s] = vs[ap * KR_AS + bp * KR_BS + li] * kf;
        }
#pragma unroll
      for (int q = 0; q < 2; ++q) acc[q] = kr_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[q] = kr_mma(ay[s], bv[q][s], acc[q]);
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) vs[(wave + 8 * h + 4 * q) * KR_AS + (lk + 4 * r) * KR_BS + li] = acc[q][r];
    }
    __syncthreads();

    // 3. Y[a][b][j] = sum_a' Ex[a][a'] T[a'][b][j] for this wavefront's b = wave + 8h + 4q
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      kr_v4d acc[2];
      double bv[2][4];
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int s = 0; s < 4; ++s) bv[q][s] = vs[(4 * s + lk) * KR_AS + (wave + 8 * h + 4 * q) * KR_BS + li];
#pragma unroll
      for (int q = 0; q < 2; ++q) acc[q] = kr_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[q] = kr_mma(ax[s], bv[q][s], acc[q]);
      if (!RIGHT) {
        // C[a n2 + b][t0 + j]: 16 consecutive columns per row
        const int c = t0 + li;
        if (F16 || c < N) {
          const double cv = csl[c];
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const int b = wave + 8 * h + 4 * q;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int a = lk + 4 * r;
              if (F16 || (a < n1 && b < n2)) {
                const int row = a * n2 + b;
                tk.C[(size_t)row * tk.ldc + c] = rsl[row] * acc[q][r] * cv;
              }
            }
          }
        }
      } else {
        // back to LDS (this wavefront's b only), written out along rows below
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r) vs[(lk + 4 * r) * KR_AS + (wave + 8 * h + 4 * q) * KR_BS + li] = acc[q][r];
      }
    }
    if (RIGHT) {
      __syncthreads();
      // C[t0 + j][a n2 + b], b fastest: along a row of C
#pragma unroll 4
      for (int u = 0; u < 16; ++u) {
        const int e = tid + 256 * u;
        const int j = e >> 8, a = (e >> 4) & 15, b = e & 15;
        const int row = t0 + j, col = a * n2 + b;
        if (F16 || (a < n1 && b < n2 && row < N))
          tk.C[(size_t)row * tk.ldc + col] =
              rsl[row] * vs[a * KR_AS + b * KR_BS + j] * csl[col];
      }
    }
    if (!more) break;
    __syncthreads();  // every read of this tile's LDS is done before the next tile is staged
    tile = nt;
    tk = tn;
    t0 = n0;
  }
}

size_t kron_shmem() { return sizeof(double) * (16 * KR_AS + 3 * 256); }  // 40 KiB: four per CU

// Grid of a launch over ntiles tiles: four workgroups per compute unit (what the LDS of one
// allows), each walking ntiles / grid tiles.
int kron_grid(int ntiles, int cus) { return std::max(1, std::min(ntiles, 4 * std::max(cus, 1))); }

// all16: every task of the launch has n1 = n2 = 16.
void launch_kron(int right, int all16, const KronTask* d_tasks, int ntasks, int ntiles, int cus, hipStream_t s) {
  if (ntasks <= 0 || ntiles <= 0) return;
  const int grid = kron_grid(ntiles, cus);
  if (right && all16) hipLaunchKernelGGL((k_kron<true, true>), dim3(grid), dim3(256), kron_shmem(), s, d_tasks, ntasks, ntiles);
  else if (right) hipLaunchKernelGGL((k_kron<true, false>), dim3(grid), dim3(256), kron_shmem(), s, d_tasks, ntasks, ntiles);
  else if (all16) hipLaunchKernelGGL((k_kron<false, true>), dim3(grid), dim3(256), kron_shmem(), s, d_tasks, ntasks, ntiles);
  else hipLaunchKernelGGL((k_kron<false, false>), dim3(grid), dim3(256), kron_shmem(), s, d_tasks, ntasks, ntiles);
}

// ---- the left products of a stabilisation block -----------------------------------------------
// Columns of X stay independent through left products, so a workgroup takes its 16 columns through all steps
// in LDS (layout and matrix-core products of k_kron<false>, the same bits): X is read and C written once per
// block instead of once per slice, and a block is one launch.  Bound by the matrix cores for many chains
// (128 matrices of 256 sites, 8 steps: 113 us against 8 x 24 us) and by the steps' latency for few
// (one 16 x 16 chain: 27 us against 8 launches of 6 us).
template <bool F16>
__global__ __launch_bounds__(256, F16 ? 4 : 3) void k_kron_chain(const KronChainTask* __restrict__ tasks, int ntasks) {
  LQMC_DYNAMIC_LDS(double, vs);
  double* const sc = vs + 16 * KR_AS;  // [2][256] scales, by the parity of the step
  const int tile = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readlane(tid >> 6, 0), li = lane & 15, lk = lane >> 4;
  const KronChainTask tk = tasks[kr_task(tasks, ntasks, tile)];
  const int t0 = (tile - tk.tile_base) * KR_T;
  const int N = F16 ? 256 : tk.N, n1 = F16 ? 16 : tk.n1, n2 = F16 ? 16 : tk.n2;
  const LQMC_GLOBAL double* X = gptr(tk.X);
  const bool pre = tk.ks != nullptr, post = tk.rs != nullptr;
  const LQMC_GLOBAL double* scg = gptr(pre ? tk.ks : tk.rs);
  const bool has = (pre || post) && tid < N;
  double nxt = has ? scg[tid] : 1.0;
  {
    double v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      int ap, bp, j;
      kr_coords<false>(tid + 256 * u, ap, bp, j);
      const bool ok = F16 || (ap < n1 && bp < n2 && t0 + j < N);
      v[u] = ldg0(X, (size_t)(ap * n2 + bp) * N + t0 + j, ok);
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
      int ap, bp, j;
      kr_coords<false>(tid + 256 * u, ap, bp, j);
      vs[ap * KR_AS + bp * KR_BS + j] = v[u];
    }
  }
  double ay[4], ax[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    ay[s] = gptr(tk.Ey)[li * 16 + 4 * s + lk];
    ax[s] = gptr(tk.Ex)[li * 16 + 4 * s + lk];
  }
  const int col = t0 + li;
  const double cv = tk.cs && col < N ? tk.cs[col] : 1.0;
#pragma unroll 1
  for (int step = 0; step < tk.steps; ++step) {
    double* const sl = sc + 256 * (step & 1);
    if (tid < N) sl[tid] = nxt;
    if (has && step + 1 < tk.steps) nxt = scg[(long)(step + 1) * tk.stride + tid];
    __syncthreads();
    // the b' direction of this wavefront's a' blocks (in place)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (!F16 && wave + 8 * h >= n1) break;
      kr_v4d acc[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) acc[q] = kr_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < 4; ++s)
        if (F16 || 4 * s < n2) {
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const int ap = wave + 8 * h + 4 * q, bp = 4 * s + lk;
            const double kf = pre && (F16 || (ap < n1 && bp < n2)) ? sl[ap * n2 + bp] : 1.0;
            acc[q] = kr_mma(ay[s], vs[ap * KR_AS + bp * KR_BS + li] * kf, acc[q]);
          }
        }
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) vs[(wave + 8 * h + 4 * q) * KR_AS + (lk + 4 * r) * KR_BS + li] = acc[q][r];
    }
    __syncthreads();
    // the a' direction of this wavefront's b (in place, or to C after the last step)
    const double cf = step == 0 ? cv : 1.0;
    const bool end = step + 1 == tk.steps;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (!F16 && wave + 8 * h >= n2) break;
      kr_v4d acc[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) acc[q] = kr_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < 4; ++s)
        if (F16 || 4 * s < n1) {
#pragma unroll
          for (int q = 0; q < 2; ++q)
            acc[q] = kr_mma(ax[s], vs[(4 * s + lk) * KR_AS + (wave + 8 * h + 4 * q) * KR_BS + li], acc[q]);
        }
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int b = wave + 8 * h + 4 * q;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int a = lk + 4 * r;
          const bool in = F16 || (a < n1 && b < n2);
          const double rf = post && in ? sl[a * n2 + b] : 1.0;
          const double v = rf * acc[q][r] * cf;
          if (!end) vs[a * KR_AS + b * KR_BS + li] = v;
          else if (in && (F16 || col < N)) gptr(tk.C)[(size_t)(a * n2 + b) * N + col] = v;
        }
      }
    }
    // the next step's first barrier orders these writes before its reads
  }
}

size_t kron_chain_shmem() { return sizeof(double) * (16 * KR_AS + 2 * 256); }

void launch_kron_chain(int all16, const KronChainTask* d_tasks, int ntasks, int ntiles, hipStream_t s) {
  if (ntasks <= 0 || ntiles <= 0) return;
  if (all16) hipLaunchKernelGGL(k_kron_chain<true>, dim3(ntiles), dim3(256), kron_chain_shmem(), s, d_tasks, ntasks);
  else hipLaunchKernelGGL(k_kron_chain<false>, dim3(ntiles), dim3(256), kron_chain_shmem(), s, d_tasks, ntasks);
}

// ---- directions of up to 32 sites -------------------------------------------------------------
// Lattices with a direction of 17 to 32 sites (N up to 1024): one workgroup per 16 columns (left) or
// rows (right) of X, a thread per fiber of either direction (kron_fiber.h).  Left tiles lie in LDS as
// [a'][b'][j], the a' blocks 16 (n2 | 1) apart, right ones as [j][k] with an odd stride, so that
// neighbouring lanes fall on different banks either way.
//
// X is read and C written once, and the contractions take 2 N^2 (n1 + n2) flops; the chain of a
// fiber's rows (scalar loads, F dependent multiply-adds) and the two memory phases of a tile, with two
// workgroups per compute unit, bound it.  64 products of 24 x 24 lattices take 178 us (left) and
// 155 us (right), 2 TB/s, where the dense 576^3 products took 565.
template <bool RIGHT>
__global__ __launch_bounds__(512) void k_kron_wide(const KronTask* __restrict__ tasks, int ntasks) {
  LQMC_DYNAMIC_LDS(double, vs);
  const int tile = xcd_grouped_block(), tid = threadIdx.x, nt = blockDim.x;
  const KronTask tk = tasks[kr_task(tasks, ntasks, tile)];
  const int t0 = (tile - tk.tile_base) * KR_T;
  const int N = tk.N, n1 = tk.n1, n2 = tk.n2;
  const int AS = 16 * (n2 | 1), LDR = N | 1;
  const LQMC_GLOBAL double* X = gptr(tk.X);
  // the scales' stored values (any valid address where there is none), so that their loads need no branch
  const LQMC_GLOBAL double* ks = gptr(tk.ks_kind != SC_NONE ? tk.ks : tk.Ex);
  const LQMC_GLOBAL double* rs = gptr(tk.rs_kind != SC_NONE ? tk.rs : tk.Ex);
  const LQMC_GLOBAL double* cs = gptr(tk.cs_kind != SC_NONE ? tk.cs : tk.Ex);
  if (RIGHT) {
    for (int k = tid; k < N; k += nt) {
      const double kf = ks[k];
      double v[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) v[j] = ldg0(X, (size_t)(t0 + j) * tk.ldx + k, t0 + j < N);
      const double kv = kr_scale_of(tk.ks_kind, kf);
#pragma unroll
      for (int j = 0; j < 16; ++j) vs[j * LDR + k] = v[j] * kv;
    }
  } else {
    const int j = tid & 15, c = t0 + j, step = nt >> 4;
    for (int k0 = tid >> 4; k0 < N; k0 += 12 * step) {
      double v[12], kf[12];
#pragma unroll
      for (int u = 0; u < 12; ++u) {
        const int k = k0 + u * step;
        v[u] = ldg0(X, (size_t)k * tk.ldx + c, k < N && c < N);
        kf[u] = ks[k < N ? k : 0];
      }
#pragma unroll
      for (int u = 0; u < 12; ++u) {
        const int k = k0 + u * step;
        if (k < N) vs[k * 16 + (k / n2) * (AS - 16 * n2) + j] = v[u] * kr_scale_of(tk.ks_kind, kf[u]);
      }
    }
  }
  __syncthreads();
#pragma unroll 1
  for (int stage = 0; stage < 2; ++stage) {  // b' with Ey, then a' with Ex
    const LQMC_CONST double* E = uniform_const(stage ? tk.Ex : tk.Ey);
    const int n = stage ? n1 : n2, other = stage ? n2 : n1;
    const int st = RIGHT ? (stage ? n2 : 1) : (stage ? AS : 16);
    for (int f = tid; f < 16 * other; f += nt) {
      const int j = f & 15, o = f >> 4;
      kf_apply<32>(vs + (RIGHT ? j * LDR + (stage ? o : o * n2) : (stage ? o * 16 : o * AS) + j), st, E, 32, n);
    }
    __syncthreads();
  }
  if (RIGHT) {
    double rf[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) rf[j] = rs[t0 + j < N ? t0 + j : 0];
#pragma unroll
    for (int j = 0; j < 16; ++j) rf[j] = kr_scale_of(tk.rs_kind, rf[j]);
    for (int k = tid; k < N; k += nt) {
      const double cv = kr_scale_of(tk.cs_kind, cs[k]);
#pragma unroll
      for (int j = 0; j < 16; ++j)
        if (t0 + j < N) gptr(tk.C)[(size_t)(t0 + j) * tk.ldc + k] = rf[j] * vs[j * LDR + k] * cv;
    }
  } else {
    const int j = tid & 15, c = t0 + j, step = nt >> 4;
    if (c < N) {
      const double cv = kr_scale_of(tk.cs_kind, cs[c]);
      for (int k0 = tid >> 4; k0 < N; k0 += 12 * step) {
        double rf[12];
#pragma unroll
        for (int u = 0; u < 12; ++u) rf[u] = rs[k0 + u * step < N ? k0 + u * step : 0];
#pragma unroll
        for (int u = 0; u < 12; ++u) {
          const int k = k0 + u * step;
          if (k < N)
            gptr(tk.C)[(size_t)k * tk.ldc + c] =
                kr_scale_of(tk.rs_kind, rf[u]) * vs[k * 16 + (k / n2) * (AS - 16 * n2) + j] * cv;
        }
      }
    }
  }
}

int kron_wide_threads(int n1, int n2) { return std::min(512, 64 * ((16 * std::max(n1, n2) + 63) / 64)); }
size_t kron_wide_shmem(int n1, int n2) {
  return sizeof(double) * 16 * (size_t)std::max(n1 * (n2 | 1), (n1 * n2) | 1);
}

void launch_kron_wide(int right, const KronTask* d_tasks, int ntasks, int ntiles, int threads, size_t shmem,
                      hipStream_t s) {
  if (ntasks <= 0 || ntiles <= 0) return;
  if (right) hipLaunchKernelGGL(k_kron_wide<true>, dim3(ntiles), dim3(threads), shmem, s, d_tasks, ntasks);
  else hipLaunchKernelGGL(k_kron_wide<false>, dim3(ntiles), dim3(threads), shmem, s, d_tasks, ntasks);
}

int kron_tiles(int N) { return (N + KR_T - 1) / KR_T; }

}  // namespace lqmc
