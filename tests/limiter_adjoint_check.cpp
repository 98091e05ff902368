// limited_slope_adj against the reverse of limited_slope written out branch by
// branch, on every triple of a small set of values: ties, uniform and opposed
// states, zeros and both magnitudes' ends, for finite bars and for infinite and
// NaN ones.  Prints the triples and the mismatches.
#include <cmath>
#include <cstdio>
#include <initializer_list>
#include <limits>

#include "../euler2d_cudafortran_amd/csrc/e2d_adjoint.hpp"

using namespace e2d;

template <class T>
static bool same(T a, T b) { return a == b || (std::isnan(a) && std::isnan(b)); }

template <class T>
static int mismatches(int& n, std::initializer_list<T> bars) {
  const T x[] = {T(-1e30), T(-2), T(-1), T(-0.5), T(-1e-20), T(0), T(1e-20), T(0.3), T(0.5), T(1), T(1.5), T(2), T(1e30)};
  int bad = 0;
  for (int st = 0; st < 2; ++st)
    for (T qm : x)
      for (T q0 : x)
        for (T qp : x)
          for (T ob : bars) {
            const T s = T(st + 1);
            const T dl = s * (q0 - qm), dr = s * (qp - q0), dc = T(0.5) * (qp - qm);
            const bool opposed = dl * dr <= T(0);
            const T lim = opposed ? T(0) : (std::fabs(dl) < std::fabs(dr) ? std::fabs(dl) : std::fabs(dr));
            T m = T(0), c = T(0), p = T(0);
            if (!(lim < std::fabs(dc))) {  // slope = dc
              m = T(-0.5) * ob;
              p = T(0.5) * ob;
            } else if (!opposed && std::fabs(dl) < std::fabs(dr)) {  // slope = dl
              c = s * ob;
              m = -s * ob;
            } else if (!opposed) {  // slope = dr
              p = s * ob;
              c = -s * ob;
            }
            T a = T(0), b = T(0), d = T(0);
            limited_slope_adj(s, qm, q0, qp, ob, a, b, d);
            bad += !(same(a, m) && same(b, c) && same(d, p));
            ++n;
          }
  return bad;
}

template <class T>
static void report(const char* name) {
  constexpr T inf = std::numeric_limits<T>::infinity(), nan = std::numeric_limits<T>::quiet_NaN();
  int n = 0, k = 0;
  const int bad = mismatches<T>(n, {T(0.7), T(-3)}), badk = mismatches<T>(k, {inf, -inf, nan});
  std::printf("%s n=%d bad=%d\n%s-nonfinite n=%d bad=%d\n", name, n, bad, name, k, badk);
}

int main() {
  report<double>("double");
  report<float>("float");
  return 0;
}
