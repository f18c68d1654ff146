// ratnodes.h -- rational approximation of x^(-1/2) on [1, kappa] (host code).
//
//   x^(-1/2) = (2/pi) int_0^inf dt / (t^2 + x)
//
// With t = sc(u | k), k'^2 = 1/kappa (Jacobi elliptic functions, modulus
// k = sqrt(1 - 1/kappa)), the poles t^2 = -x, x in [1, kappa], move to the
// line Im u = K' and the integrand becomes even about u = 0 and u = K, so
// the midpoint rule on [0, K] converges like exp(-2 pi K' N / K)
// (about exp(-2 pi^2 N / log(16 kappa))):
//
//   x^(-1/2) ~= sum_j w_j / (x + s_j),   u_j = (j - 1/2) K / N,
//   s_j = sc^2(u_j),   w_j = (2 K / (pi N)) dn(u_j) nc^2(u_j).
//
// For a symmetric positive definite A with spectrum in [m, m kappa],
// A^(-1/2) = m^(-1/2) (A/m)^(-1/2) ~= sum_j sqrt(m) w_j (A + m s_j I)^-1.
//
// sn, cn, dn come from the arithmetic-geometric mean (descending Landen)
// method; for u > K/2 the quarter-period reflection u -> K - u keeps cn and
// the square of sc accurate when k is close to 1.
#pragma once

#include <algorithm>
#include <cmath>
#include <limits>
#include <vector>

namespace lk {
namespace rat {

template <typename T>
constexpr T kPi = (T)3.141592653589793238462643383279502884L;

// complete elliptic integral K(k) = pi / (2 AGM(1, k'))
template <typename T>
inline T ellipk_c(T kc) {
  T a = 1, b = kc;
  for (int i = 0; i < 64 && std::fabs(a - b) > std::numeric_limits<T>::epsilon() / 16 * a; ++i) {
    const T an = (a + b) / 2;
    b = std::sqrt(a * b);
    a = an;
  }
  return kPi<T> / (2 * a);
}

// sn, cn, dn of u for modulus k (k' = kc), AGM method
template <typename T>
inline void ellipj(T u, T k, T kc, T* sn, T* cn, T* dn) {
  T a[40], c[40];
  a[0] = 1;
  T b = kc;
  c[0] = k;
  int n = 0;
  while (n < 38 && std::fabs(c[n]) > std::numeric_limits<T>::epsilon() / 16) {
    a[n + 1] = (a[n] + b) / 2;
    c[n + 1] = (a[n] - b) / 2;
    b = std::sqrt(a[n] * b);
    ++n;
  }
  T phi = std::ldexp(a[n] * u, n);
  T phi_prev = phi;
  for (int i = n; i >= 1; --i) {
    phi_prev = phi;
    phi = (phi + std::asin(c[i] * std::sin(phi) / a[i])) / 2;
  }
  *sn = std::sin(phi);
  *cn = std::cos(phi);
  *dn = n >= 1 ? std::cos(phi) / std::cos(phi_prev - phi) : T(1);
}

// nodes for [1, kappa] with n points: s[j] = sc^2(u_j), w[j]; computed in T
template <typename T>
inline void nodes_in(T kappa, int n, T* s, T* w) {
  const T kc = 1 / std::sqrt(kappa);
  const T k = std::sqrt((1 - kc) * (1 + kc));
  const T K = ellipk_c(kc);
  for (int j = 0; j < n; ++j) {
    const T u = (j + T(0.5)) * K / n;
    T sc2, dnc2;
    if (u <= K / 2) {
      T sn, cn, dn;
      ellipj(u, k, kc, &sn, &cn, &dn);
      sc2 = (sn / cn) * (sn / cn);
      dnc2 = dn / (cn * cn);
    } else {
      // u = K - v: sn = cn(v)/dn(v), cn = k' sn(v)/dn(v), dn = k'/dn(v)
      T sn, cn, dn;
      ellipj(K - u, k, kc, &sn, &cn, &dn);
      const T r = cn / (kc * sn);               // sc(u)
      sc2 = r * r;
      dnc2 = (kc / dn) * (dn / (kc * sn)) * (dn / (kc * sn));   // dn(u) nc(u)^2
    }
    s[j] = sc2;
    w[j] = 2 * K / (kPi<T> * n) * dnc2;
  }
}
inline void nodes(double kappa, int n, double* s, double* w) { nodes_in<double>(kappa, n, s, w); }

// largest relative error of the n-point approximation over [1, kappa]
// (log-spaced samples; the error is a smooth function of log x), summed in T
template <typename T>
inline double max_rel_err_in(double kappa, int n, const double* s, const double* w,
                             int samples) {
  T e = 0;
  for (int i = 0; i <= samples; ++i) {
    const T x = std::exp(std::log((T)kappa) * i / samples);
    T acc = 0;
    for (int j = 0; j < n; ++j) acc += w[j] / (x + s[j]);
    e = std::fmax(e, std::fabs(acc * std::sqrt(x) - 1));
  }
  return (double)e;
}
inline double max_rel_err(double kappa, int n, const double* s, const double* w,
                          int samples = 1500) {
  return max_rel_err_in<double>(kappa, n, s, w, samples);
}

// fewest nodes that can meet tol: the error falls like
// exp(-2 pi^2 n / log(16 kappa)); two below, so that no smaller n does
inline int fewest(double kappa, double tol) {
  return std::max(2, (int)(-std::log(tol) * std::log(16.0 * kappa) / (2.0 * M_PI * M_PI)) - 2);
}

// smallest n in nmin..nmax meeting tol on [1, kappa]; fills s, w; returns n
// or -1
inline int choose(double kappa, double tol, int nmax, double* s, double* w, int nmin = 2) {
  for (int n = nmin; n <= nmax; ++n) {
    nodes(kappa, n, s, w);
    if (max_rel_err(kappa, n, s, w) <= tol) return n;
  }
  return -1;
}

// the same for a tolerance at the rounding of the values themselves: nodes
// and error in extended precision, the nodes rounded once
inline int choose_fine(double kappa, double tol, int nmax, double* s, double* w) {
  std::vector<long double> ls((size_t)nmax), lw((size_t)nmax);
  for (int n = std::min(fewest(kappa, tol), nmax); n <= nmax; ++n) {
    nodes_in<long double>(kappa, n, ls.data(), lw.data());
    for (int j = 0; j < n; ++j) { s[j] = (double)ls[(size_t)j]; w[j] = (double)lw[(size_t)j]; }
    if (max_rel_err_in<long double>(kappa, n, s, w, 200) <= tol) return n;
  }
  return -1;
}

}  // namespace rat
}  // namespace lk
