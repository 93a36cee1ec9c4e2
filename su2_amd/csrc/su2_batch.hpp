// su2_batch.hpp -- descriptors and launchers of the batched-ensemble kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <vector>

#include "su2_launch.hpp"

namespace su2k {

// one lattice of the batch (device copy)
struct BLat {
  Geo geo;
  int group;      // 0 U(1), 1 SU(2)
  int kind;       // integrator id: 0 leapfrog, 6 omf2
  int npairs;     // number of "P then U" pairs; tick npairs is the final momentum step
  int cur;        // arena holding the configuration at the start of the trajectory
  int fin;        // arena holding the last link update
  int tile0, ntiles;    // site tiles (sums, momenta, restore)
  int ltile0, nltiles;  // link tiles (MD ticks): one per (site tile, mu)
  int zs;               // z-shuffle path allowed (64 % L_fastest == 0, V % tile == 0)
  int spec;             // 4, 3: SU(2) in that dimension through the specialised step body (md_su2_core); 0: generic
  long uoff;      // byte offset of the lattice's links in every link arena
  long poff;      // element offset of its momenta in the momentum arena
  double coef;    // beta / Nc
  double dtau;    // tau / nsteps
  uint64_t seed;  // Philox key of its momenta
};

struct BArenas {
  char *U[3];
  void *P;
};

// integrator pair k of lattice l: (P coefficient, U coefficient) in units of dtau
__device__ inline void pair_coef(int kind, int k, double &cp, double &cu) {
  if (kind == 6) {  // omf2 (integrator.hh:83-115): P(l) [U(1/2) P(1-2l) U(1/2) P(2l)]... P(l)
    const double lam = 0.1938;
    cp = (k == 0) ? lam : ((k & 1) ? 1. - 2. * lam : 2. * lam);
    cu = 0.5;
  } else {  // leapfrog (integrator.hh:26-50): P(1/2) U(1) [P(1) U(1)]... P(1/2)
    cp = (k == 0) ? 0.5 : 1.0;
    cu = 1.0;
  }
}
__device__ inline double final_coef(int kind) { return kind == 6 ? 0.1938 : 0.5; }
// tick of lattice L: the step's coefficients and the arenas it reads and writes
__device__ inline void batch_tick_coef(const BLat &L, int tick, int flags, FusedCoef &c, int &rd,
                                       int &wr) {
  const int a0 = L.cur, a1 = (L.cur + 1) % 3, a2 = (L.cur + 2) % 3;
  c.coef = L.coef;
  c.w_t = 1.0;
  c.w_s = 1.0;
  c.flags = flags;
  if (tick != L.npairs) {
    double cp, cu;
    pair_coef(L.kind, tick, cp, cu);
    c.ep = cp * L.dtau;
    c.eu = cu * L.dtau;
    rd = (tick == 0) ? a0 : ((tick & 1) ? a1 : a2);
    wr = (tick & 1) ? a2 : a1;
  } else {
    c.ep = final_coef(L.kind) * L.dtau;
    rd = L.npairs == 0 ? a0 : (((L.npairs - 1) & 1) ? a2 : a1);
    wr = rd;
  }
}

// ltiles: (lattice, site_start * 4 + mu): those of the specialised SU(2)
// lattices in d = 4 ([0, n4)), then in d = 3 ([n4, n4 + n3)), then the rest;
// partial rows are nltiles long.  One launch of at most `grid` blocks for one part
// (0: d = 4, 1: d = 3, 2: the rest), so that each part has its own register budget.
// active: the number of the part's leading tiles that belong to lattices still running
// at this tick (each part's lattices are ordered by step count, longest first).
void launch_batch_tick(int prec, const BLat *lats, const int2 *ltiles, int nltiles, int n4, int n3,
                       const BArenas &ar, int tick, int flags, double *partials, int grid,
                       int block, hipStream_t st, int part, int active);
// The ticks of the specialised d = 4 part with the shared-plaquette step
// (su2_batch_plq.hip).  A plan: tiles (lattice, block of the lattice's layout) in the
// lattices' order and the layouts (PlqGeo, one per lattice of the batch).
struct BatchPlqPlan {
  unsigned threads = 0, lds = 0;
  std::vector<char> geos;
  std::vector<int2> tiles;
};
// tick t runs the first `count` tiles of plan `plan` (-1: its link tiles).  The slices
// of a chunk are chosen for the lattices still running: a new plan whenever their sites
// fell below three quarters of the last plan's.
struct BatchPlqTicks {
  struct Tick {
    int plan = -1, count = 0;
  };
  std::vector<BatchPlqPlan> plans;
  std::vector<Tick> tick;
};
// `part`: the part's lattices, those with more steps first.  A tick whose running
// lattices are too few, do not all fit the layout or leave too many lanes idle keeps
// the link tiles.
void plan_batch_plq(int prec, int ncu, const std::vector<BLat> &lat, const std::vector<size_t> &part,
                    int maxpairs, BatchPlqTicks &out);
void launch_batch_plq(int prec, const BLat *lats, const void *geos, const int2 *tiles, int count,
                      int rowlen, const BArenas &ar, int tick, int flags, double *partials,
                      unsigned threads, unsigned lds, hipStream_t st);
void launch_batch_plaq(int prec, const BLat *lats, const int2 *tiles, int ntiles, const BArenas &ar,
                       int use_final, int row, int rowlen, double *partials, int grid, int block,
                       hipStream_t st);
void launch_batch_restore(int prec, const BLat *lats, const int2 *tiles, int ntiles,
                          const BArenas &ar, int grid, int block, hipStream_t st);
void launch_batch_momenta(int prec, const BLat *lats, const int2 *tiles, int ntiles,
                          const BArenas &ar, const uint64_t *traj, int grid, int block,
                          hipStream_t st);
void launch_batch_reduce(const BLat *lats, int nlat, const double *partials, int rowlen,
                         double *out, hipStream_t st);

}  // namespace su2k
