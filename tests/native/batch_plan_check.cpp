// The plan of the batch's shared-plaquette ticks (plan_batch_plq) on the host.  Input: the
// precision, then per member Lx Ly Lz Lt npairs.  Checks of every tick: its tiles are
// those of the running members, every block of each exactly once, no other's; a member
// has at least as many link tiles as blocks.  Prints per tick the plan, its tiles and
// the running sites.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <numeric>

#include "../../su2_amd/csrc/su2_batch_plq.hip"

using namespace su2k;

int main(int argc, char **argv) {
  if (argc < 7 || (argc - 2) % 5 != 0) return 2;
  const int prec = atoi(argv[1]);
  std::vector<BLat> lat;
  int maxpairs = 0;
  for (int i = 2; i < argc; i += 5) {
    BLat b{};
    b.geo.L[1] = atoi(argv[i]);
    b.geo.L[2] = atoi(argv[i + 1]);
    b.geo.L[3] = atoi(argv[i + 2]);
    b.geo.L[0] = atoi(argv[i + 3]);
    b.geo.nd = 4;
    b.geo.V = b.geo.L[0] * b.geo.L[1] * b.geo.L[2] * b.geo.L[3];
    b.npairs = atoi(argv[i + 4]);
    b.nltiles = 4 * ((b.geo.V + 255) / 256);
    maxpairs = std::max(maxpairs, b.npairs);
    lat.push_back(b);
  }
  std::vector<size_t> part(lat.size());
  std::iota(part.begin(), part.end(), (size_t)0);
  std::stable_sort(part.begin(), part.end(),
                   [&](size_t x, size_t y) { return lat[x].npairs > lat[y].npairs; });
  BatchPlqTicks out;
  plan_batch_plq(prec, 256, lat, part, maxpairs, out);
  if ((int)out.tick.size() != maxpairs + 1) return 3;
  for (int t = 0; t <= maxpairs; ++t) {
    long run = 0;
    for (const BLat &b : lat)
      if (b.npairs >= t) run += b.geo.V;
    const auto tk = out.tick[t];
    printf("%d %d %d %ld\n", t, tk.plan, tk.count, run);
    if (tk.plan < 0) continue;
    if (tk.plan >= (int)out.plans.size()) return 4;
    const BatchPlqPlan &p = out.plans[tk.plan];
    if (tk.count < 1 || tk.count > (int)p.tiles.size()) return 5;
    const PlqGeo *geo = (const PlqGeo *)p.geos.data();
    std::vector<std::vector<int>> seen(lat.size());
    for (int i = 0; i < tk.count; ++i) {
      const int2 tl = p.tiles[i];
      if (lat[tl.x].npairs < t) return 6;
      seen[tl.x].push_back(tl.y);
    }
    for (size_t l = 0; l < lat.size(); ++l) {
      if (lat[l].npairs < t) continue;
      const uint32_t nb = plq_blocks(geo[l]);
      if (seen[l].size() != nb || (int)nb > lat[l].nltiles) return 7;
      std::sort(seen[l].begin(), seen[l].end());
      for (uint32_t k = 0; k < nb; ++k)
        if (seen[l][k] != (int)k) return 8;
      if (plq_threads(geo[l]) > p.threads || plq_lds<PlqSU2<double>, 4>(geo[l]) == 0) return 9;
    }
  }
  return 0;
}
