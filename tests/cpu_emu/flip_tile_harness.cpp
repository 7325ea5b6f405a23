// CPU build of the register-tile flip (k_flip_tile): one slice of every chain against the rank-1
// kernel on the same state and uniforms -- the same decisions and ratios, field and G to 1e-12,
// the same exp(V) tables, counters and (on slice 0) measurement; every access in bounds.
// usage: flip_tile_harness N L nchains t measure gscale [class]   (class: a form covering more sites)
#include "hip_cpu_shim.h"
#include "../../latticeqmc_amd/csrc/flip.hip"
#include "../../latticeqmc_amd/csrc/flip_tile.hip"

#include <cstdio>
#include <cstdlib>
#include <random>

using namespace lqmc;

template <typename T>
static T* dalloc(size_t n) { return static_cast<T*>(std::calloc(n ? n : 1, sizeof(T))); }

struct Batch {
  std::vector<ChainDev> ch;
  std::vector<ChainState> st;
};

static Batch make(int N, int L, int nch, double gscale) {
  Batch b;
  b.ch.resize(nch);
  b.st.resize(nch);
  std::memset(b.st.data(), 0, sizeof(ChainState) * nch);
  std::mt19937_64 rng(7);
  std::uniform_real_distribution<double> U(-0.3, 0.3);
  for (int c = 0; c < nch; ++c) {
    const int n = std::max(1, N - c), l = std::max(1, L - c);  // uneven chains
    const size_t n2 = (size_t)n * n;
    ChainDev& d = b.ch[c];
    std::memset(&d, 0, sizeof d);
    d.N = n; d.L = l; d.lam = 0.6;
    d.e1m = std::exp(-0.6); d.e1p = std::exp(0.6); d.e2p = std::exp(1.2); d.e2m = std::exp(-1.2);
    d.seed = 1234 + c;
    d.field = dalloc<int8_t>((size_t)n * l);
    for (size_t e = 0; e < (size_t)n * l; ++e) d.field[e] = (rng() & 1) ? 1 : -1;
    d.ev = dalloc<double>(2 * (size_t)n * l);
    d.evi = dalloc<double>(2 * (size_t)n * l);
    double* g = dalloc<double>(2 * n2);
    for (size_t e = 0; e < 2 * n2; ++e) g[e] = gscale * U(rng) / n + ((e % n2) / n == (e % n2) % n ? 0.5 : 0.0);
    d.G = g;
    d.Gacc = dalloc<double>(2 * n2); d.Glast = dalloc<double>(2 * n2); d.Sacc = dalloc<double>(n2);
    d.hop = dalloc<double>(n2);
    d.tr_ratio = dalloc<double>((size_t)n * l); d.tr_acc = dalloc<uint8_t>((size_t)n * l);
    d.obs_cap = 8;
    d.obs = dalloc<double>(24);
  }
  return b;
}

template <int T, int WR>
static void run(FlipArgs a, int nch) {
  constexpr int threads = 128 * WR * WR, NP = 8 * T * WR;
  const size_t sh = sizeof(double) * (9 * NP + std::max(threads, NP)) + sizeof(int) * (NP + NP / 8);
  emu_launch(nch, threads, sh, [&] { k_flip_tile<T, WR>(a); });
}

int main(int argc, char** argv) {
  if (argc < 7) return 2;
  const int N = atoi(argv[1]), L = atoi(argv[2]), nch = atoi(argv[3]), t = atoi(argv[4]), measure = atoi(argv[5]);
  const double gscale = atof(argv[6]);
  Batch x = make(N, L, nch, gscale), y = make(N, L, nch, gscale);
  std::vector<int> list(nch);
  for (int c = 0; c < nch; ++c) list[c] = nch - 1 - c;
  FlipArgs a{x.ch.data(), x.st.data(), t, measure, 1, 1, 1, 1, nullptr, nch, 0, 0, list.data()};
  switch (argc > 7 ? atoi(argv[7]) : flip_tile_class(N)) {
    case 0: run<2, 1>(a, nch); break;
    case 1: run<4, 1>(a, nch); break;
    case 2: run<3, 2>(a, nch); break;
    case 3: run<4, 2>(a, nch); break;
    case 4: run<5, 2>(a, nch); break;
    case 5: run<6, 2>(a, nch); break;
    case 6: run<7, 2>(a, nch); break;
    case 7: run<8, 2>(a, nch); break;
    default: return 2;
  }
  FlipArgs b{y.ch.data(), y.st.data(), t, measure, 1, 1, 1, 0};
  emu_launch(nch, 256, sizeof(double) * (4 * (size_t)N + 256), [&] { k_flip_rank1<double>(b); });
  double dg = 0.0, dr = 0.0, dm = 0.0;
  int diff = 0;
  unsigned long long acc = 0;
  auto far = [](double p, double q) { const double d = std::fabs(p - q); return d == d ? d : 1e300; };
  for (int c = 0; c < nch; ++c) {
    const ChainDev &p = x.ch[c], &q = y.ch[c];
    const size_t n2 = (size_t)p.N * p.N, nl = (size_t)p.N * p.L;
    for (size_t e = 0; e < 2 * n2; ++e) {
      dg = std::max(dg, far(static_cast<double*>(p.G)[e], static_cast<double*>(q.G)[e]));
      dm = std::max(dm, std::max(far(p.Gacc[e], q.Gacc[e]), far(p.Glast[e], q.Glast[e])));
    }
    for (size_t e = 0; e < n2; ++e) dm = std::max(dm, far(p.Sacc[e], q.Sacc[e]));
    for (int e = 0; e < 24; ++e) dm = std::max(dm, far(p.obs[e], q.obs[e]));
    for (size_t e = 0; e < nl; ++e) {
      diff += p.field[e] != q.field[e] || p.tr_acc[e] != q.tr_acc[e];
      dr = std::max(dr, far(p.tr_ratio[e], q.tr_ratio[e]));
    }
    for (size_t e = 0; e < 2 * nl; ++e) diff += p.ev[e] != q.ev[e] || p.evi[e] != q.evi[e];
    diff += x.st[c].accepted != y.st[c].accepted || x.st[c].attempted != y.st[c].attempted ||
            x.st[c].sweep != y.st[c].sweep || x.st[c].measured != y.st[c].measured || x.st[c].flags || y.st[c].flags;
    acc += x.st[c].accepted;
  }
  std::printf("N=%d accepted %llu |dG| %.2e ratio %.2e measured %.2e differences %d\n", N, acc, dg, dr, dm, diff);
  const bool ok = dg <= 1e-12 && dr <= 1e-11 && dm <= 1e-11 && diff == 0;
  std::printf(ok ? "ok\n" : "FAIL\n");
  return ok ? 0 : 1;
}
