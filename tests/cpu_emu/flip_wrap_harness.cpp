// CPU build of the register-tile flip with wraps (k_flip_tile<.., true>): slices t .. t + slices - 1 of
// every chain in one launch against the same kernel without wraps, slice by slice, with the dense wrap
// G <- E^-1 V^-1 G V E on the host between them -- the same decisions, fields, tables and counters, G and
// the measurement to rounding; every access in bounds.
// usage: flip_wrap_harness n1 n2 L nchains t slices measure [class]
#include "hip_cpu_shim.h"
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
  std::vector<std::vector<double>> E, Ei;  // dense E and E^-1 of every chain
};

// exp(+-0.1 * ring hopping) of n sites, by its series
static std::vector<double> factor(int n, double x) {
  std::vector<double> k(n * n, 0.0), e(n * n, 0.0), p(n * n, 0.0);
  for (int i = 0; i < n; ++i) { k[i * n + (i + 1) % n] += x; k[((i + 1) % n) * n + i] += x; e[i * n + i] = p[i * n + i] = 1.0; }
  for (int m = 1; m < 30; ++m) {
    std::vector<double> q(n * n, 0.0);
    for (int i = 0; i < n; ++i) for (int j = 0; j < n; ++j) for (int r = 0; r < n; ++r) q[i * n + j] += p[i * n + r] * k[r * n + j] / m;
    p = q;
    for (int e2 = 0; e2 < n * n; ++e2) e[e2] += p[e2];
  }
  // an asymmetric pair: D E and E^-1 D^-1, so that a transposed factor shows
  for (int i = 0; i < n; ++i) for (int j = 0; j < n; ++j) e[i * n + j] *= x > 0 ? 1.0 + 0.01 * i : 1.0 / (1.0 + 0.01 * j);
  return e;
}

static Batch make(int n1, int n2, int L, int nch) {
  Batch b;
  b.ch.resize(nch); b.st.resize(nch); b.E.resize(nch); b.Ei.resize(nch);
  std::memset(b.st.data(), 0, sizeof(ChainState) * nch);
  std::mt19937_64 rng(7);
  std::uniform_real_distribution<double> U(-0.3, 0.3);
  for (int c = 0; c < nch; ++c) {
    const int m1 = std::max(2, n1 - c), n = m1 * n2, l = std::max(1, L - c);  // uneven chains
    const size_t nn = (size_t)n * n;
    ChainDev& d = b.ch[c];
    std::memset(&d, 0, sizeof d);
    d.N = n; d.L = l; d.lam = 0.6;
    d.e1m = std::exp(-0.6); d.e1p = std::exp(0.6); d.e2p = std::exp(1.2); d.e2m = std::exp(-1.2);
    d.seed = 1234 + c;
    d.field = dalloc<int8_t>((size_t)n * l);
    for (size_t e = 0; e < (size_t)n * l; ++e) d.field[e] = (rng() & 1) ? 1 : -1;
    d.ev = dalloc<double>(2 * (size_t)n * l);
    d.evi = dalloc<double>(2 * (size_t)n * l);
    double* g = dalloc<double>(2 * nn);
    for (size_t e = 0; e < 2 * nn; ++e) g[e] = U(rng) / n + ((e % nn) / n == (e % nn) % n ? 0.5 : 0.0);
    d.G = g;
    d.Gacc = dalloc<double>(2 * nn); d.Glast = dalloc<double>(2 * nn); d.Sacc = dalloc<double>(nn);
    d.hop = dalloc<double>(nn);
    d.tr_ratio = dalloc<double>((size_t)n * l); d.tr_acc = dalloc<uint8_t>((size_t)n * l);
    d.obs_cap = 8;
    d.obs = dalloc<double>(24);
    d.kn1 = m1; d.kn2 = n2;
    double* kr = dalloc<double>(8 * 256);
    b.E[c].resize(nn); b.Ei[c].resize(nn);
    for (int inv = 0; inv < 2; ++inv) {
      const std::vector<double> ex = factor(m1, inv ? -0.1 : 0.1), ey = factor(n2, inv ? -0.1 : 0.1);
      for (int i = 0; i < m1; ++i) for (int j = 0; j < m1; ++j) kr[(2 * inv) * 256 + i * 16 + j] = kr[(4 + 2 * inv) * 256 + j * 16 + i] = ex[i * m1 + j];
      for (int i = 0; i < n2; ++i) for (int j = 0; j < n2; ++j) kr[(2 * inv + 1) * 256 + i * 16 + j] = kr[(5 + 2 * inv) * 256 + j * 16 + i] = ey[i * n2 + j];
      auto& e = inv ? b.Ei[c] : b.E[c];
      for (int i = 0; i < n; ++i) for (int j = 0; j < n; ++j) e[(size_t)i * n + j] = ex[(i / n2) * m1 + j / n2] * ey[(i % n2) * n2 + j % n2];
    }
    d.kr = kr;
  }
  return b;
}

template <int T, int WR>
static void run(FlipArgs a, int nch) {
  constexpr int threads = 128 * WR * WR;
  if (a.slices) emu_launch(nch, threads, ft_shmem<T, WR>(true), [&] { k_flip_tile<T, WR, true>(a); });
  else emu_launch(nch, threads, ft_shmem<T, WR>(false), [&] { k_flip_tile<T, WR>(a); });
}

static void flip(int cls, FlipArgs a, int nch) {
  switch (cls) {
    case 0: run<2, 1>(a, nch); break;
    case 1: run<4, 1>(a, nch); break;
    case 2: run<3, 2>(a, nch); break;
    case 3: run<4, 2>(a, nch); break;
    case 4: run<5, 2>(a, nch); break;
    case 5: run<6, 2>(a, nch); break;
    case 6: run<7, 2>(a, nch); break;
    case 7: run<8, 2>(a, nch); break;
    default: std::abort();
  }
}

static void dense_wrap(Batch& b, int c, int t) {
  const ChainDev& d = b.ch[c];
  const int n = d.N, l = d.L - 1 - t;
  std::vector<double> w((size_t)n * n), z((size_t)n * n);
  for (int s = 0; s < 2; ++s) {
    double* G = static_cast<double*>(d.G) + (size_t)s * n * n;
    const double *ev = d.ev + (size_t)s * n * d.L + (size_t)l * n, *evi = d.evi + (size_t)s * n * d.L + (size_t)l * n;
    for (int i = 0; i < n; ++i) for (int j = 0; j < n; ++j) {
      double v = 0.0;
      for (int k = 0; k < n; ++k) v += b.Ei[c][(size_t)i * n + k] * evi[k] * G[(size_t)k * n + j];
      w[(size_t)i * n + j] = v * ev[j];
    }
    for (int i = 0; i < n; ++i) for (int j = 0; j < n; ++j) {
      double v = 0.0;
      for (int k = 0; k < n; ++k) v += w[(size_t)i * n + k] * b.E[c][(size_t)k * n + j];
      z[(size_t)i * n + j] = v;
    }
    std::copy(z.begin(), z.end(), G);
  }
}

int main(int argc, char** argv) {
  if (argc < 8) return 2;
  const int n1 = atoi(argv[1]), n2 = atoi(argv[2]), L = atoi(argv[3]), nch = atoi(argv[4]), t0 = atoi(argv[5]);
  const int slices = atoi(argv[6]), measure = atoi(argv[7]);
  const int cls = argc > 8 ? atoi(argv[8]) : flip_tile_class(n1 * n2);
  Batch x = make(n1, n2, L, nch), y = make(n1, n2, L, nch);
  FlipArgs a{x.ch.data(), x.st.data(), t0, measure, 1, 1, 1, 1, nullptr, nch, 0, 0, nullptr, slices};
  flip(cls, a, nch);
  for (int t = t0; t < t0 + slices; ++t) {
    FlipArgs b{y.ch.data(), y.st.data(), t, measure, 1, 1, 1, 1, nullptr, nch, 0, 0, nullptr, 0};
    flip(cls, b, nch);
    for (int c = 0; c < nch; ++c)
      if (t < y.ch[c].L) dense_wrap(y, c, t);
  }
  double dg = 0.0, dr = 0.0, dm = 0.0;
  int diff = 0;
  auto far = [](double p, double q) { const double d = std::fabs(p - q); return d == d ? d : 1e300; };
  for (int c = 0; c < nch; ++c) {
    const ChainDev &p = x.ch[c], &q = y.ch[c];
    const size_t nn = (size_t)p.N * p.N, nl = (size_t)p.N * p.L;
    for (size_t e = 0; e < 2 * nn; ++e) {
      dg = std::max(dg, far(static_cast<double*>(p.G)[e], static_cast<double*>(q.G)[e]));
      dm = std::max(dm, std::max(far(p.Gacc[e], q.Gacc[e]), far(p.Glast[e], q.Glast[e])));
    }
    for (size_t e = 0; e < nn; ++e) dm = std::max(dm, far(p.Sacc[e], q.Sacc[e]));
    for (int e = 0; e < 24; ++e) dm = std::max(dm, far(p.obs[e], q.obs[e]));
    for (size_t e = 0; e < nl; ++e) {
      diff += p.field[e] != q.field[e] || p.tr_acc[e] != q.tr_acc[e];
      dr = std::max(dr, far(p.tr_ratio[e], q.tr_ratio[e]));
    }
    for (size_t e = 0; e < 2 * nl; ++e) diff += p.ev[e] != q.ev[e] || p.evi[e] != q.evi[e];
    diff += x.st[c].accepted != y.st[c].accepted || x.st[c].attempted != y.st[c].attempted ||
            x.st[c].sweep != y.st[c].sweep || x.st[c].measured != y.st[c].measured || x.st[c].flags || y.st[c].flags;
  }
  std::printf("%d x %d |dG| %.2e ratio %.2e measured %.2e differences %d\n", n1, n2, dg, dr, dm, diff);
  const bool ok = dg <= 1e-11 && dr <= 1e-10 && dm <= 1e-10 && diff == 0;
  std::printf(ok ? "ok\n" : "FAIL\n");
  return ok ? 0 : 1;
}
