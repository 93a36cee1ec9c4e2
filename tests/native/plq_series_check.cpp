// The sine / cosine series of su2_md_plq.hpp against 80-bit arithmetic on the host:
// largest errors of cos a and sin(a)/a as functions of x = a^2 (cos_sinc_fp64) for x
// up to 1 and up to 12, and of the reduced sine and cosine of angles up to 3e4 and beyond, in units of 2^-53.
#include <cmath>
#include <cstdio>

#include "../../su2_amd/csrc/su2_md_plq.hpp"

using namespace su2k;

int main() {
  const long double u = 0x1p-53L;
  long double ec[2] = {}, es[2] = {}, rc[2] = {}, rs[2] = {};
  auto top = [](long double &m, long double e) {
    e = fabsl(e);
    if (!(e <= m)) m = e;
  };
  // x over (0, 12], dense below 1.5
  for (int i = 1; i <= 600000; ++i) {
    const double x = i <= 400000 ? 1.5 * i / 400000.0 + 1e-9 : 1.5 + 10.5 * (i - 400000) / 200000.0;
    double c, s;
    cos_sinc_fp64(x, c, s);
    const long double a = sqrtl((long double)x);
    top(ec[x > 1.0], c - cosl(a));
    top(es[x > 1.0], s - sinl(a) / a);
  }
  // angles up to 3e4, to 1e8 and to 4e14
  for (double f : {1.0, 3333.33, 1.3e10})
    for (int i = -400000; i <= 400000; ++i) {
      const double a = i * 0.0750000001 * f;
      int j;
      const double r = plq_reduce(a, j);
      double c, s;
      plq_sincos(r, c, s);
      plq_quadrant(j, c, s);
      top(rc[f > 1.0], c - cosl((long double)a));
      top(rs[f > 1.0], s - sinl((long double)a));
    }
  printf("%.4Lf %.4Lf %.4Lf %.4Lf %.4Lf %.4Lf %.4Lf %.4Lf\n", ec[0] / u, es[0] / u, ec[1] / u,
         es[1] / u, rc[0] / u, rs[0] / u, rc[1] / u, rs[1] / u);
  return 0;
}
