// Replays the launch layout of the shared-plaquette step (su2_md_plq.hpp) on
// the host: for the extents t, x, y, z and the number of blocks resident on each of 256 CUs given
// on the command line, every site is taken by exactly one active thread of one
// slice walk, the neighbour offsets are the periodic lexicographic ones, and
// the threads that a site exchanges with through LDS hold its neighbours.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../su2_amd/csrc/su2_md_plq.hpp"

using namespace su2k;

int main(int argc, char **argv) {
  if (argc != 7) return 2;
  const int nd = atoi(argv[1]);
  const int L[4] = {atoi(argv[2]), atoi(argv[3]), atoi(argv[4]), atoi(argv[5])};
  const int slots = atoi(argv[6]);
  const int V = L[0] * L[1] * L[2] * L[3];
  PlqGeo g;
  if (!make_plq_rows(L, nd, V, g) || !make_plq_chunks(slots, 256, g)) {
    printf("not applicable\n");
    return 0;
  }
  const uint32_t nb = plq_blocks(g), nt = plq_threads(g);
  if (nt > (uint32_t)PLQ_NT || nt % 64 != 0) return 3;
  const int slots_lds = (int)nt + L[nd - 1];
  const int str[4] = {L[1] * L[2] * L[3], L[2] * L[3], L[3], 1};
  auto nbr = [&](int s, int d, int by) {
    const int c = (s / str[d]) % L[d];
    return s + ((c + by + L[d]) % L[d] - c) * str[d];
  };
  const int R = nd - 2, Z = nd - 1;
  std::vector<int> seen(V, 0);
  for (uint32_t b = 0; b < nb; ++b) {
    std::vector<PlqSite> f(nt);
    for (uint32_t i = 0; i < nt; ++i) {
      f[i] = plq_site(g, b, nb, i, nt);
      if (f[i].t0 != f[0].t0 || f[i].t1 != f[0].t1) return 4;  // uniform walk
      // every lane addresses sites of the lattice and slots of the block
      if (f[i].o3 < 0 || f[i].o3 >= g.vol3 || f[i].t0 < 0 || f[i].t1 > L[0] ||
          f[i].t0 >= f[i].t1)
        return 5;
      if (f[i].lur < 0 || f[i].lur >= slots_lds || (f[i].rin && f[i].lur >= (int)nt)) return 6;
      if (f[i].ldr >= (int)nt || f[i].luz < 0 || f[i].luz >= (int)nt || f[i].ldz < 0 ||
          f[i].ldz >= (int)nt)
        return 7;
    }
    std::vector<int> halo(slots_lds, -1);
    for (uint32_t i = 0; i < nt; ++i)
      if (f[i].active && !f[i].rin) {
        if (halo[f[i].lur] >= 0) return 8;  // one writer per halo slot
        halo[f[i].lur] = f[i].o3 + f[i].ur;
      }
    for (uint32_t i = 0; i < nt; ++i) {
      const int o = f[i].o3;
      if (nd == 4 && (o + f[i].ux != nbr(o, 1, 1) || o + f[i].dx != nbr(o, 1, -1))) return 9;
      if (o + f[i].ur != nbr(o, R, 1) || o + f[i].dr != nbr(o, R, -1)) return 10;
      if (o + f[i].uz != nbr(o, Z, 1) || o + f[i].dz != nbr(o, Z, -1)) return 11;
      if (!f[i].active) continue;
      if (f[i].rin ? (!f[f[i].lur].active || f[f[i].lur].o3 != nbr(o, R, 1))
                   : halo[f[i].lur] != nbr(o, R, 1))
        return 12;
      if (f[i].ldr >= 0 && (!f[f[i].ldr].active || f[f[i].ldr].o3 != nbr(o, R, -1))) return 13;
      if (!f[f[i].luz].active || f[f[i].luz].o3 != nbr(o, Z, 1)) return 14;
      if (!f[f[i].ldz].active || f[f[i].ldz].o3 != nbr(o, Z, -1)) return 15;
      for (int t = f[i].t0; t < f[i].t1; ++t) ++seen[t * g.vol3 + o];
    }
  }
  for (int s = 0; s < V; ++s)
    if (seen[s] != 1) return 16;
  printf("ok rows/block %d threads %u Tc %d blocks %u\n", g.rpb, nt, g.Tc, nb);
  return 0;
}
