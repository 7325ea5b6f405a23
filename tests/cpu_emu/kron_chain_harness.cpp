// CPU build of k_kron_chain: the left products of a block of slices in one launch against k_kron, one launch
// per product -- the same bits; two tasks of different sizes, one scaled before (ks), one after (rs) each step,
// every access in bounds.
// usage: kron_chain_harness n1 n2 n1b n2b steps
#include "hip_cpu_shim.h"
#include "../../latticeqmc_amd/csrc/kron.hip"

#include <cstdio>
#include <cstdlib>
#include <random>

using namespace lqmc;

int main(int argc, char** argv) {
  if (argc < 6) return 2;
  const int steps = atoi(argv[5]);
  std::mt19937_64 rng(11);
  std::normal_distribution<double> g(0.0, 1.0);
  std::uniform_real_distribution<double> u(0.5, 2.0);
  int diff = 0, base = 0;
  std::vector<KronChainTask> tasks(2);
  std::vector<double> ex[2], ey[2], X[2], C[2], sc[2], cs[2];
  for (int t = 0; t < 2; ++t) {
    const int n1 = atoi(argv[1 + 2 * t]), n2 = atoi(argv[2 + 2 * t]), N = n1 * n2;
    ex[t].assign(256, 0.0); ey[t].assign(256, 0.0);
    for (int a = 0; a < n1; ++a) for (int b = 0; b < n1; ++b) ex[t][a * 16 + b] = g(rng);
    for (int a = 0; a < n2; ++a) for (int b = 0; b < n2; ++b) ey[t][a * 16 + b] = g(rng);
    X[t].resize((size_t)N * N); C[t].assign((size_t)N * N, 7.0); sc[t].resize((size_t)N * steps); cs[t].resize(N);
    for (auto& v : X[t]) v = g(rng);
    for (auto& v : sc[t]) v = u(rng);
    for (auto& v : cs[t]) v = u(rng);
    // the first task walks its scales upwards, the second downwards
    double* s0 = t ? sc[t].data() + (size_t)N * (steps - 1) : sc[t].data();
    tasks[t] = KronChainTask{X[t].data(), C[t].data(), ex[t].data(), ey[t].data(), t ? nullptr : s0, t ? s0 : nullptr,
                             t ? cs[t].data() : nullptr, N, n1, n2, steps, t ? -N : N, base};
    base += kron_tiles(N);
  }
  const bool all16 = tasks[0].N == 256 && tasks[1].N == 256 && tasks[0].n1 == 16 && tasks[1].n1 == 16;
  if (all16) emu_launch(base, 256, kron_chain_shmem(), [&] { k_kron_chain<true>(tasks.data(), 2); });
  else emu_launch(base, 256, kron_chain_shmem(), [&] { k_kron_chain<false>(tasks.data(), 2); });
  for (int t = 0; t < 2; ++t) {
    const KronChainTask& c = tasks[t];
    std::vector<double> w = X[t], z(w.size());
    for (int s = 0; s < steps; ++s) {
      KronTask k{};
      k.X = w.data(); k.C = z.data(); k.Ex = c.Ex; k.Ey = c.Ey;
      k.rs = c.rs ? c.rs + (long)s * c.stride : nullptr; k.rs_kind = c.rs ? SC_PLAIN : SC_NONE;
      k.ks = c.ks ? c.ks + (long)s * c.stride : nullptr; k.ks_kind = c.ks ? SC_PLAIN : SC_NONE;
      k.cs = c.cs; k.cs_kind = c.cs && s == 0 ? SC_PLAIN : SC_NONE;
      k.N = c.N; k.n1 = c.n1; k.n2 = c.n2; k.ldx = k.ldc = c.N;
      const int nt = kron_tiles(c.N);
      if (all16) emu_launch(nt, 256, kron_shmem(), [&] { k_kron<false, true>(&k, 1, nt); });
      else emu_launch(nt, 256, kron_shmem(), [&] { k_kron<false, false>(&k, 1, nt); });
      w.swap(z);
    }
    for (size_t e = 0; e < w.size(); ++e) diff += !(w[e] == C[t][e]);
  }
  std::printf("%s: %d entries differ\n", diff ? "FAIL" : "ok", diff);
  return diff != 0;
}
