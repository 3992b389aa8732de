// Host check: the fluxes of a face along an axis (RoeFlux::flux_axis,
// NewtonianViscousFlux::compute_flux_axis) equal the general forms
// (flux_frame, compute_flux) for finite states, values compared with ==
// (an exact zero may differ in sign), and where the general inviscid flux is
// not finite the axis form is not either.  FP64 and FP32, all axes, both
// signs, states from rest to supersonic, velocities with exact zeros and tiny
// values.  Usage: axis_flux_check [count]; exits non-zero on any mismatch.
#include <math.h>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <limits>
#include "physics.hpp"
using namespace ma;
static uint64_t s = 0x9E3779B97F4A7C15ull;
static uint64_t nxt() { s += 0x9E3779B97F4A7C15ull; uint64_t z = s; z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull; z = (z ^ (z >> 27)) * 0x94D049BB133111EBull; return z ^ (z >> 31); }
static double uni(double a, double b) { return a + (b - a) * (double)(nxt() >> 11) / 9007199254740992.0; }
template <class T> void state(T* v) {
  v[0] = T(std::exp(uni(-7, 3)));
  v[4] = T(uni(50, 3000));
  for (int k = 1; k < 4; ++k) {
    const int r = (int)(nxt() % 8);
    v[k] = T(r == 0 ? 0.0 : r == 1 ? uni(-1e-30, 1e-30) : uni(-900, 900));
  }
}
template <int D, class T> long axis(long n) {
  long bad = 0;
  const RoeFlux roe{};
  const NewtonianViscousFlux visc{0.72};
  for (long i = 0; i < n; ++i) {
    T l[5], r[5], a[3] = {T(0), T(0), T(0)}, F[5], G[5], g[5][3];
    state(l);
    if (nxt() % 5) state(r);
    else for (int k = 0; k < 5; ++k) r[k] = l[k];
    if (i % 50 == 0) {
      const T odd[3] = {std::numeric_limits<T>::quiet_NaN(), std::numeric_limits<T>::infinity(), T(-1)};
      ((nxt() & 1) ? l : r)[nxt() % 5] = odd[nxt() % 3];
    }
    for (auto& q : g) for (T& x : q) x = nxt() % 6 ? T(uni(-1e5, 1e5)) : T(0);
    a[D] = T(std::ldexp(uni(1, 2), -(int)(nxt() % 40)) * ((nxt() & 1) ? 1 : -1));
    inviscid_flux(roe, l, r, F, frame_from_area_t<T>(a));
    inviscid_flux_axis<D>(roe, l, r, G, a[D]);
    T V[5], f[5], h[5];
    for (int k = 0; k < 5; ++k) V[k] = T(0.5) * (l[k] + r[k]);
    visc.compute_flux(g, V, a, f);
    visc.template compute_flux_axis<D, T>(g, V, a[D], h);
    bool same = true, finite = true;
    for (int k = 0; k < 5; ++k) finite = finite && std::isfinite(F[k]) && std::isfinite(f[k]);
    for (int k = 0; k < 5; ++k) {
      const T x = F[k] - f[k], y = G[k] - h[k];
      same = same && (finite ? F[k] == G[k] && f[k] == h[k] : x == y || (std::isnan(x) && std::isnan(y)));
    }
    if (!same && ++bad < 5) printf("mismatch axis %d at %ld\n", D, i);
  }
  return bad;
}
template <class T> long run(long n) {
  const long bad = axis<0, T>(n) + axis<1, T>(n) + axis<2, T>(n);
  printf("%s: n=%ld mismatches=%ld\n", sizeof(T) == 8 ? "double" : "float", 3 * n, bad);
  return bad;
}
int main(int argc, char** argv) {
  const long n = argc > 1 ? std::atol(argv[1]) : 2000000L;
  return run<double>(n) + run<float>(n) ? 1 : 0;
}
