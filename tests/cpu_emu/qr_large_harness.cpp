// Numerical and bounds check of the QR of large matrices (k_ql_*, N up to 640) in a
// CPU build, as qr_harness.cpp checks the smaller ones: graded W = M diag(d), W = Q diag(D) V''
// and W P = Q diag(D) R' column-relative, Q^T Q = I, R' upper triangular with unit-modulus pivots.
// A matrix with a zero column must raise the zero-pivot flag and nothing else.
// usage: qr_large_harness N decades seed [zero]
#include "hip_cpu_shim.h"
#include "../../latticeqmc_amd/csrc/qr_large.hip"

#include <cstdio>
#include <cstdlib>
#include <random>
#include <string>

using namespace lqmc;

int main(int argc, char** argv) {
  if (argc < 4) return 2;
  const int N = atoi(argv[1]);
  const double decades = atof(argv[2]);
  const bool zero = argc > 4 && std::string(argv[4]) == "zero";
  std::mt19937_64 rng(atoi(argv[3]));
  std::normal_distribution<double> g(0.0, 1.0);
  std::uniform_real_distribution<double> uni(-0.5, 0.5);
  const size_t n2 = (size_t)N * N;
  std::vector<double> W0(n2), d(N);
  for (int c = 0; c < N; ++c) d[c] = std::pow(10.0, decades * uni(rng));
  for (int r = 0; r < N; ++r)
    for (int c = 0; c < N; ++c) W0[(size_t)r * N + c] = zero && c == N / 2 ? 0.0 : g(rng) * d[c];
  auto alloc = [&](size_t n) { return static_cast<double*>(std::malloc(n * 8)); };
  double *W = alloc(n2), *Q = alloc(n2), *D = alloc(N), *A = alloc(n2), *Tt = alloc(16 * (N + 16));
  int* perm = static_cast<int*>(std::malloc(N * sizeof(int)));
  ChainState st[2] = {};
  // a second task of one column, and a block count for a larger matrix than either
  double one[4] = {};  // W, Q, D, A
  std::vector<double> tt1(16 * 17);
  const int n = 2, nmax = N + 17, nb64 = (nmax + 63) / 64, nbr = (nmax + QL_ROWS - 1) / QL_ROWS, nb32 = (nmax + 31) / 32;
  double rec[2] = {0.0, 0.0}, orth = 0.0, low = 0.0, dia = 0.0;
  size_t nonfinite = 0;
  for (int pass = 0; pass < 2; ++pass) {  // without and with the pivot order
    std::copy(W0.begin(), W0.end(), W);
    QrTask t{W, Q, D, A, pass ? perm : nullptr, Tt, N, 0};
    one[0] = -3.0;
    QrTask tasks[2] = {t, QrTask{one, one + 1, one + 2, one + 3, nullptr, tt1.data(), 1, 1}};
    emu_launch(n * nb64, 256, 256 * sizeof(double), [&] { k_ql_norms(tasks, nb64, st); });
    emu_launch(n * nb64, 256, ql_order_shmem(), [&] { k_ql_order(tasks, nb64); });
    emu_launch(n * nbr, 256, ql_rows_shmem(nmax), [&] { k_ql_gather(tasks, nbr); });
    for (int P = 0; 16 * P < nmax; ++P) {
      const int rest = nmax - 16 * (P + 1), nblk = 1 + (P > 0 && rest > 0 ? (rest + 31) / 32 : 0);
      emu_launch(8 * nblk, QL_THREADS, ql_step_shmem(), [&] { k_ql_step(tasks, n, nblk, P, st); });
    }
    emu_launch(n * nbr, 256, ql_rows_shmem(nmax), [&] { k_ql_out(tasks, nbr); });
    emu_launch(n * nb32, QL_THREADS, ql_formq_shmem(), [&] { k_ql_formq(tasks, nb32); });
    if (std::fabs(one[1] * one[2] * one[0] + 3.0) > 1e-15) return 1;
    for (int c = 0; c < N; ++c) {
      double cn = 0.0, en = 0.0;
      for (int r = 0; r < N; ++r) {
        double s = 0.0;
        for (int k = 0; k < N; ++k) s += Q[(size_t)r * N + k] * D[k] * W[(size_t)k * N + c];
        const double w0 = W0[(size_t)r * N + (pass ? perm[c] : c)];
        cn += w0 * w0;
        en += (s - w0) * (s - w0);
      }
      if (cn > 0.0) rec[pass] = std::max(rec[pass], std::sqrt(en / cn));
    }
    for (size_t e = 0; e < n2; ++e) nonfinite += !std::isfinite(Q[e]) + !std::isfinite(W[e]);
  }
  for (int i = 0; i < N; ++i)
    for (int j = 0; j < N; ++j) {
      double s = 0.0;
      for (int k = 0; k < N; ++k) s += Q[(size_t)k * N + i] * Q[(size_t)k * N + j];
      orth = std::max(orth, std::fabs(s - (i == j ? 1.0 : 0.0)));
      if (j < i) low = std::max(low, std::fabs(W[(size_t)i * N + j]));
      if (j == i && !zero) dia = std::max(dia, std::fabs(std::fabs(W[(size_t)i * N + j]) - 1.0));
    }
  std::printf("N=%d decades=%g recon %.2e %.2e orth %.2e lower %.1e |diag|-1 %.1e flags %u nonfinite %zu\n", N, decades,
              rec[0], rec[1], orth, low, dia, st[0].flags, nonfinite);
  const bool ok = rec[0] < 1e-12 && rec[1] < 1e-12 && orth < 1e-12 && low == 0.0 && dia < 1e-12 && nonfinite == 0 &&
                  st[0].flags == (zero ? 2u : 0u);
  std::printf(ok ? "ok\n" : "FAIL\n");
  return ok ? 0 : 1;
}
