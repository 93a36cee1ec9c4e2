// The chunk choice of the shared-plaquette step (su2_md_plq.hpp) against a plain sum over
// the rounds, and its time for a lattice long in t: it is made at every launch.
#include <chrono>
#include <cstdio>

#include "../../su2_amd/csrc/su2_md_plq.hpp"

using namespace su2k;

static int plain_choice(const PlqGeo &g, int percu, int cus) {
  const int waves = (g.rpb * g.L[g.nd - 1] + 63) / 64;
  double cost = 1e300;
  int best = 1;
  for (int Tc = 1; Tc <= g.L[0]; ++Tc) {
    const int nc = (g.L[0] + Tc - 1) / Tc;
    double c = 0.0;
    for (long left = (long)g.nb3 * nc; left > 0; left -= (long)percu * cus) {
      const long b = std::min<long>((left + cus - 1) / cus, percu);
      c += (Tc + 0.35) * (2.0 + (double)(b * waves));
    }
    if (c < cost * 0.999) {
      cost = c;
      best = Tc;
    }
  }
  return best;
}

int main() {
  for (int nd : {3, 4})
    for (int t : {1, 2, 7, 16, 27, 48, 96, 131, 1000})
      for (int y : {1, 3, 9, 18, 48})
        for (int z : {2, 5, 16, 24, 61, 128})
          for (int x : {1, 4, 20, 48})
            for (int percu : {1, 2, 4, 8}) {
              const int L[4] = {t, nd == 4 ? x : y * x, nd == 4 ? y : z, nd == 4 ? z : 1};
              PlqGeo g;
              if (!make_plq_rows(L, nd, L[0] * L[1] * L[2] * L[3], g)) continue;
              if (!make_plq_chunks(percu, 256, g)) return 1;
              if (g.Tc != plain_choice(g, percu, 256)) {
                printf("%d: %d %d %d %d, %d: %d against %d\n", nd, L[0], L[1], L[2], L[3], percu,
                       g.Tc, plain_choice(g, percu, 256));
                return 2;
              }
            }
  // the share of lanes that hold a site, planes y z
  const struct {
    int y, z;
    double fill;
  } planes[] = {{3, 3, 9.0 / 64}, {4, 4, 16.0 / 64}, {1, 2, 2.0 / 64}, {9, 9, 81.0 / 128},
                {32, 32, 1.0},    {24, 24, 1.0},     {8, 8, 1.0},      {20, 20, 400.0 / 448},
                {5, 61, 305.0 / 320}};
  for (const auto &q : planes) {
    const int L[4] = {16, 4, q.y, q.z};
    PlqGeo g;
    if (!make_plq_rows(L, 4, 64 * q.y * q.z, g)) return 5;
    if (std::fabs(plq_fill(g) - q.fill) > 1e-12) {
      printf("%d %d: %f against %f\n", q.y, q.z, plq_fill(g), q.fill);
      return 6;
    }
    // 64 planes: small enough to take either way, 64 t slices of 64 are not
    if (!plq_full(g)) return 7;
    const int M[4] = {64, 64, q.y, q.z};
    if (!make_plq_rows(M, 4, 4096 * q.y * q.z, g) || plq_full(g) != (q.fill >= 0.5)) return 8;
  }
  const int L[4] = {1 << 20, 4, 8, 1};
  const auto t0 = std::chrono::steady_clock::now();
  long sum = 0;
  for (int i = 0; i < 1000; ++i) {
    PlqGeo g;
    if (!make_plq_rows(L, 3, L[0] * 32, g) || !make_plq_chunks(8, 256, g)) return 3;
    sum += g.Tc;
  }
  const double us =
      std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count() / 1000;
  printf("ok %.1f us a plan, Tc %ld\n", us, sum / 1000);
  return us < 1000.0 ? 0 : 4;
}
