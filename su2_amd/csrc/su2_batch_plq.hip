// su2_batch_plq.hip -- one MD tick of the batch's SU(2) lattices in d = 4 with the shared-plaquette step (su2_md_plq.hpp).
//
// The link tiles of su2_batch.hip form every staple product once per link; this
// step forms a plaquette once for its four links and needs half the link requests.
// Lattices of different extents share a launch: a tile is one block of its own
// lattice's layout, blocks have the threads and LDS of the largest layout and the
// waves past their tile's own end at once (an ended wave does not count at a barrier).
//
// Bound as the single lattice's step: latency and issue.  The 32 lattices of 8^4,
// 12^4 and 16^4 of the mixed ensemble (1.05 M sites, FP32, beside the d = 3 and U(1)
// ticks): 63.3 -> 59.6 us on the average of a trajectory, the first tick, whose sums cost 24
// spilled registers in FP32, 94 -> 92 us (with 2 waves per SIMD and no spills a trajectory
// takes as long).  The same step for the d = 3 part (273000 sites)
// took 25 us where the link tiles take 20: not built.
#include "su2_batch.hpp"
#include "su2_md_plq.hpp"

namespace su2k {

template <class G, bool FIRST>
__global__ __launch_bounds__(PLQ_NT, plq_occ<G>()) void k_batch_plq(
    const BLat *__restrict__ lats, const PlqGeo *__restrict__ geos, const int2 *__restrict__ tiles,
    int rowlen, BArenas ar, int tick, int flags, double *__restrict__ partials) {
  using T = typename G::T;
  using link = typename G::link;
  constexpr int ND = 4;
  extern __shared__ __align__(16) char smem[];
  const int2 tl = tiles[xcd_block(blockIdx.x, gridDim.x)];
  const BLat &L = lats[tl.x];
  PlqGeo g = geos[tl.x];
  g.nd = ND;  // known to the compiler: no indexing at run time
  const int nt = (int)plq_threads(g);
  if (__builtin_amdgcn_readfirstlane((int)threadIdx.x) >= nt) return;  // whole waves
  const PlqSite f = plq_site_at(g, (uint32_t)tl.y, threadIdx.x, (uint32_t)nt);
  FusedCoef c{};
  int rd, wr;
  batch_tick_coef(L, tick, flags, c, rd, wr);
  const link *ui = (const link *)(ar.U[rd] + L.uoff);
  link *uo = (link *)(ar.U[wr] + L.uoff);
  T *P = (T *)ar.P + L.poff;
  double sums[3] = {0.0, 0.0, 0.0};
  const bool final_p = tick == L.npairs;
  if constexpr (FIRST) {
    plq_step<G, ND, true, true, false, 0>(f, nt, smem, ui, uo, (const T *)P, P, g, c, sums);
  } else {
    if (!final_p) plq_step<G, ND, true, false, false, 0>(f, nt, smem, ui, uo, (const T *)P, P, g, c, sums);
    else plq_step<G, ND, false, true, false, 0>(f, nt, smem, ui, uo, (const T *)P, P, g, c, sums);
  }
  if (FIRST || final_p) {
    // the lattice's partials have an entry for each of its link tiles, at least
    // as many as it has blocks here: this block's sum and zeros
    const double v = plq_block_sums(sums, nt, smem);
    const int k = (int)threadIdx.x, nb = (int)(g.nb3 * g.nchunk);
    if (FIRST ? k < 2 : k == 2) {
      double *row = partials + (size_t)k * rowlen + L.ltile0;
      row[tl.y] = v;
      for (int i = tl.y + nb; i < L.nltiles; i += nb) row[i] = 0.0;
    }
  }
}

// the layouts and chunks of the first n lattices of `part`
template <class G>
static bool plan_part(int ncu, const std::vector<BLat> &lat, const std::vector<size_t> &part,
                      size_t n, BatchPlqPlan &p) {
  std::vector<PlqGeo> geo(lat.size());
  p = BatchPlqPlan{};
  const std::vector<size_t> run(part.begin(), part.begin() + n);
  int maxT = 1;
  for (size_t l : run) {
    PlqGeo &g = geo[l];
    if (!make_plq_rows(lat[l].geo.L, 4, lat[l].geo.V, g)) return false;
    p.threads = std::max(p.threads, plq_threads(g));
    p.lds = std::max(p.lds, (unsigned)plq_lds<G, 4>(g));
    maxT = std::max(maxT, g.L[0]);
  }
  // slices per chunk for all lattices together: the cost of make_plq_chunks
  const int percu = std::max(1, std::min(plq_occ<G>() * 4 * 64 / (int)p.threads, (int)(160 * 1024 / p.lds)));
  double cost = 1e300;
  int best = 1;
  for (int Tc = 1; Tc <= maxT; ++Tc) {
    double nb = 0.0, waves = 0.0, c = 0.0;
    for (size_t l : run) {
      const PlqGeo &g = geo[l];
      const double n = (double)g.nb3 * ((g.L[0] + Tc - 1) / Tc);
      nb += n;
      waves += n * plq_threads(g) / 64;
    }
    waves /= nb;
    for (double left = nb; left > 0.0 && c < cost; left -= (double)percu * ncu)
      c += (Tc + 0.35) * (2.0 + std::min(std::ceil(left / ncu), (double)percu) * waves);
    if (c < cost * 0.999) {
      cost = c;
      best = Tc;
    }
  }
  for (size_t l : run) {
    PlqGeo &g = geo[l];
    g.Tc = std::min(best, g.L[0]);
    // longer chunks where a small lattice would have more blocks than entries for
    // their sums
    while (g.Tc < g.L[0] && g.nb3 * ((g.L[0] + g.Tc - 1) / g.Tc) > lat[l].nltiles) ++g.Tc;
    g.nchunk = (g.L[0] + g.Tc - 1) / g.Tc;
    if ((uint64_t)g.nb3 * g.nchunk * g.nb3 >= (1ull << 32)) return false;
    g.mnyb = fast_div_magic((uint32_t)g.nyb);
    g.mnb3 = fast_div_magic((uint32_t)g.nb3);
    const int nb = (int)plq_blocks(g);
    if (nb > lat[l].nltiles) return false;
    for (int b = 0; b < nb; ++b) p.tiles.push_back(int2{(int)l, b});
  }
  p.geos.assign((const char *)geo.data(), (const char *)(geo.data() + geo.size()));
  return true;
}

// Running sites from which a tick takes these tiles, and the lanes that may go with a
// site.  Batches of equal members on one GPU, a trajectory of 20 steps (these tiles /
// link tiles): FP64 full waves 32 x 8^4 423 / 571 us, 4 x 16^4 697 / 962, three quarters full
// 16 x 12^4 917 / 1214, 24 x 7^4 336 / 336; FP32 full waves 32 x 8^4 292 / 307, 8 x 16^4 748 / 831,
// three quarters full 8 x 12^4 410 / 359, 32 x 12^4 1118 / 1076, 64 x 7^4 410 / 381, 16 x 10^4 392 /
// 355 us.  The mixed ensemble of 8^4, 12^4 and 16^4 has 1.08 lanes to a site.
static double min_sites(int prec) { return prec == 0 ? 32768 : 98304; }
static double max_lanes(int prec) { return prec == 0 ? 1.5 : 1.2; }

void plan_batch_plq(int prec, int ncu, const std::vector<BLat> &lat, const std::vector<size_t> &part,
                    int maxpairs, BatchPlqTicks &out) {
  out.plans.clear();
  out.tick.assign(maxpairs + 1, BatchPlqTicks::Tick{});
  // of the first n lattices: sites, lanes, and those the layout does not take
  std::vector<double> sites(1, 0.0), lanes(1, 0.0);
  std::vector<int> bad(1, 0);
  for (size_t l : part) {
    PlqGeo g;
    const bool ok = make_plq_rows(lat[l].geo.L, 4, lat[l].geo.V, g) && g.nb3 <= lat[l].nltiles;
    sites.push_back(sites.back() + lat[l].geo.V);
    lanes.push_back(lanes.back() + (ok ? (double)g.nb3 * plq_threads(g) * g.L[0] : 0.0));
    bad.push_back(bad.back() + (ok ? 0 : 1));
  }
  size_t n = part.size();
  double tried = 0.0;  // sites at the last attempt at a plan, and whether there is one for them
  bool have = false;
  std::vector<int> end;
  for (int t = 0; t <= maxpairs; ++t) {
    while (n > 0 && lat[part[n - 1]].npairs < t) --n;
    if (n == 0 || sites[n] < min_sites(prec)) break;
    if (bad[n] > 0 || lanes[n] > max_lanes(prec) * sites[n]) continue;
    if (tried == 0.0 || sites[n] < 0.75 * tried) {
      tried = sites[n];
      BatchPlqPlan p;
      have = prec == 0 ? plan_part<PlqSU2<double>>(ncu, lat, part, n, p)
                       : plan_part<PlqSU2<float>>(ncu, lat, part, n, p);
      if (have) {
        end.assign(lat.size(), 0);
        for (size_t i = 0; i < p.tiles.size(); ++i) end[p.tiles[i].x] = (int)i + 1;
        out.plans.push_back(std::move(p));
      }
    }
    if (have) out.tick[t] = {(int)out.plans.size() - 1, end[part[n - 1]]};
  }
}

void launch_batch_plq(int prec, const BLat *lats, const void *geos, const int2 *tiles, int count,
                      int rowlen, const BArenas &ar, int tick, int flags, double *partials,
                      unsigned threads, unsigned lds, hipStream_t st) {
#define SU2_BPLQ(T, F)                                                                           \
  hipLaunchKernelGGL((k_batch_plq<PlqSU2<T>, F>), dim3(count), dim3(threads), lds, st, lats,     \
                     (const PlqGeo *)geos, tiles, rowlen, ar, tick, flags, partials)
  if (prec == 0) {
    if (tick == 0) SU2_BPLQ(double, true);
    else SU2_BPLQ(double, false);
  } else {
    if (tick == 0) SU2_BPLQ(float, true);
    else SU2_BPLQ(float, false);
  }
#undef SU2_BPLQ
}

}  // namespace su2k
