// EMFs and face fluxes of the default build's solvers (mhd_device.hpp) on the CPU, for states at
// the ends of their range.  Built once as it is and once with PPK_KEEP_ROUNDING, which takes the
// reference's expressions for the Alfven speeds and star states; both print the same edges.
//
// Usage: edge_emf vanishing N   field components of 0 and of 1e-100 .. 1e-320 beside ordinary ones
//        edge_emf cold N        gas at the pressure floor moving along x at up to 1e7: the sound speed
//                               is lost in u, so that the wave speeds along x fall together
//        edge_emf stream N      the same, a dense stream running into gas at the density floor:
//                               the fastest wave falls on the contact
// prints per line the EMF in double and in float; for stream the 8 fluxes of HLLD
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "mhd_device.hpp"

using namespace ppk;

namespace {

unsigned long long seed = 12345;
double uniform(double a, double b) {
  seed = seed * 6364136223846793005ull + 1442695040888963407ull;
  return a + (b - a) * double(seed >> 11) * 0x1p-53;
}
// 0, an ordinary value or one of 10^-lo .. 10^-hi, either sign
double field(double lo, double hi) {
  const double k = uniform(0.0, 1.0), s = uniform(-1.0, 1.0) < 0 ? -1.0 : 1.0;
  if (k < 0.2) return 0.0;
  return s * (k < 0.3 ? uniform(0.01, 1.0) : std::pow(10.0, -uniform(lo, hi)));
}

DevParams params() {
  DevParams p{};
  p.gamma0 = 5.0 / 3.0;
  p.smallr = p.smallc = 1e-10;
  p.smallp = p.smallc * p.smallc / p.gamma0;
  return p;
}

template <class R>
St<R> state(double u0, double lo, double hi) {
  St<R> q;
  q[ID] = R(uniform(0.05, 2.0));
  q[IP] = R(uniform(0.05, 2.0));
  for (int v : {IU, IV, IW}) q[v] = R(u0 * uniform(-1.0, 1.0));
  for (int v : {IA, IB, IC}) q[v] = R(field(lo, hi));
  return q;
}

template <class R>
double vanishing(double lo, double hi, double u0) {
  St<R> q[4];
  for (auto &s : q) s = state<R>(u0, lo, hi);
  return double(compute_emf<EMFZ>(q[0], q[1], q[2], q[3], params()));
}

// gas at the pressure floor
St<double> cold(double rho, double u, double b) {
  const DevParams p = params();
  St<double> q;
  q[ID] = rho;
  q[IP] = rho * p.smallp;
  q[IU] = u;
  q[IV] = uniform(-1.0, 1.0);
  q[IW] = uniform(-1.0, 1.0);
  for (int v : {IA, IB, IC}) q[v] = b * uniform(-1.0, 1.0);
  return q;
}

}  // namespace

int main(int argc, char **argv) {
  if (argc < 3) return 2;
  const int n = std::atoi(argv[2]);
  for (int i = 0; i < n; ++i) {
    if (!std::strcmp(argv[1], "cold")) {
      const double u = std::pow(10.0, uniform(6.5, 7.5)), b = i % 2 ? 1e-12 : 0.0;
      St<double> q[4];
      for (auto &s : q) s = cold(uniform(0.5, 2.0), u, b);
      std::printf("%.17g 0\n", compute_emf<EMFZ>(q[0], q[1], q[2], q[3], params()));
      continue;
    }
    if (!std::strcmp(argv[1], "stream")) {
      const double u = std::pow(10.0, uniform(6.5, 7.5));
      St<double> l = cold(1e8, u, 0.0), r = cold(1e-10, -u, 0.0), f;
      riemann_hlld(l, r, f, params());
      for (int v = 0; v < 8; ++v) std::printf("%.17g ", f[v]);
      std::printf("\n");
      continue;
    }
    const double u0 = i % 2 ? 0.5 : 0.0;  // resting gas: the region around u = 0
    const double d = vanishing<double>(100.0, 320.0, u0);
    const double f = vanishing<float>(12.0, 45.0, u0);
    std::printf("%.17g %.9g\n", d, f);
  }
  return 0;
}
