// su2_plq.hip -- launches of the shared-plaquette step (su2_md_plq.hpp).
#include "su2_md_plq.hpp"

namespace su2k {

namespace {

constexpr int CUS = 256;  // MI355X

// resident blocks on a CU: registers leave room for 8 waves (SU(2) FP64, 2 per
// SIMD), 12 (SU(2) FP32) or 16 (U(1)), LDS for 160 KB
template <class G> int plq_percu(const PlqGeo &g) {
  const int waves = (int)plq_threads(g) / 64;
  const int lds = (int)(g.nd == 4 ? plq_lds<G, 4>(g) : plq_lds<G, 3>(g));
  const int fit = G::NM == 1 ? 16 : sizeof(typename G::T) == 8 ? 8 : 12;
  return std::max(1, std::min(fit / waves, 160 * 1024 / lds));
}

// The layout, or false where the staple steps are taken instead.  Below 32768
// (FP64) and 98304 sites (FP32) those are as fast or faster: a launch is bound by
// its chain of memory round trips, of which this step has two more (FP64 step
// with events, this / staples: 12^4 10.2 / 9.8, 16^4 12.3 / 13.1, d = 3 32^3 8.5 /
// 8.7 us; FP32: 16^4 10.5 / 9.7, d = 3 48^3 8.8 / 9.1 us; U(1) FP64 12^4 8.9 / 8.1, 16^4
// 9.1 / 11.1, d = 3 32^3 6.8 / 7.1 us, FP32 16^4 8.1 / 7.7, 20 18 15 27 10.2 / 11.4 us).
// FP32 SU(2) in d = 4 counts 140000 sites' worth of full lanes (x y z t, steps of a
// trajectory: 18^4 13.4 / 11.7, 40 10 10 40 16.4 / 14.6, 20^4 14.6 / 14.9, 24^4 24.1 / 24.9,
// 28^4 41.2 / 45.6 us; 24 24 24 32 33.8 / 30.9 and 32^4 58.4 / 55.5 are its two slower ones).
//
// Rows that leave lanes idle (few sites per x plane) cost as much as full ones.  The
// least share of lanes with a site, this / staples on both sides of the line (x y z t):
// SU(2) FP64 0.6: 15 5 planes 0.59 11.8 / 11.2, 5 5 0.39 34.9 / 33.6, 3 3 0.14 56.2 / 26.1, 1 2
// 0.03 89 / 48 us; 9 9 0.63 14.1 / 16.9, 9 5 0.70 9.4 / 11.4 us.  SU(2) FP32 0.7: 9 9 51.9 /
// 48.6, 6 7 0.66 51.7 / 49.3; 7 7 0.77 52.9 / 58.1, 11 11 0.95 56.3 / 72.3 us.  U(1) FP64 0.35:
// 4 4 0.25 10.6 / 8.9, 25.7 / 25.5; 5 5 7.8 / 8.7, 27.5 / 37.2 us; FP32 0.5: 5 6 0.47 9.3 / 8.9;
// 6 6 0.56 9.4 / 9.9, 9 9 13.2 / 18.1 us.
bool plq_geo_for(int group, int prec, const Geo &geo, PlqGeo &g) {
  const int pref = plq_pref();
  if (pref == 0 || !make_plq_rows(geo.L, geo.nd, geo.V, g)) return false;
  if (pref < 0) {
    const double fill = plq_fill(g);
    if (geo.V < (prec == 0 ? 32768 : 98304)) return false;
    if (group == 1 && prec == 1 && geo.nd == 4 && geo.V * fill < 140000) return false;
    if (fill < (group == 1 ? (prec == 0 ? 0.6 : 0.7) : (prec == 0 ? 0.35 : 0.5))) return false;
  }
  const int percu = group == 1 ? (prec == 0 ? plq_percu<PlqSU2<double>>(g) : plq_percu<PlqSU2<float>>(g))
                               : (prec == 0 ? plq_percu<PlqU1<double>>(g) : plq_percu<PlqU1<float>>(g));
  return make_plq_chunks(percu, CUS, g);
}

template <class G, int ND, bool W, bool ACC, bool GEN, int NT, class UI, class UO>
void go(UI ui, UO uo, const FusedLaunch &L, const PlqGeo &g, hipStream_t st) {
  using T = typename G::T;
  const unsigned lds = (unsigned)plq_lds<G, ND>(g);
  hipLaunchKernelGGL((k_md_plq<G, ND, W, ACC, GEN, NT, UI, UO>), dim3(plq_blocks(g)),
                     dim3(plq_threads(g)), lds, st, ui, uo, (const T *)L.P,
                     (T *)(L.Pout ? L.Pout : L.P), g, L.c, L.partials, L.pstride);
}

template <class G, int ND, class UI, class UO>
void go_wa(UI ui, UO uo, const FusedLaunch &L, const PlqGeo &g, bool nt, hipStream_t st) {
  const bool acc = (L.c.flags & F_ACCUM) != 0;
#define SU2_GO(W, A, GN)                                       \
  do {                                                         \
    if (nt) go<G, ND, W, A, GN, 2, UI, UO>(ui, uo, L, g, st);  \
    else go<G, ND, W, A, GN, 0, UI, UO>(ui, uo, L, g, st);     \
  } while (0)
  if (L.Uout) {
    if (acc && L.gen) SU2_GO(true, true, true);
    else if (acc) SU2_GO(true, true, false);
    else SU2_GO(true, false, false);
  } else {
    if (acc) SU2_GO(false, true, false);
    else SU2_GO(false, false, false);
  }
#undef SU2_GO
}

}  // namespace

bool plq_ok(int group, int prec, const Geo &geo, int flags) {
  PlqGeo g;
  return !(flags & (F_ROUND | F_R32L | F_R32P)) && plq_geo_for(group, prec, geo, g);
}

int plq_partials(int group, int prec, const Geo &geo) {
  PlqGeo g;
  return plq_geo_for(group, prec, geo, g) ? (int)plq_blocks(g) : 0;
}

bool launch_plq(int group, int prec, const FusedLaunch &L, hipStream_t st) {
  if (L.c.flags & (F_ROUND | F_R32L | F_R32P)) return false;
  if (L.gen && !(genfuse_pref() && L.Uout && (L.c.flags & F_ACCUM))) return false;
  if (L.in_half && L.Uout && !L.out_half) return false;  // half -> record steps are not built
  PlqGeo g;
  if (!plq_geo_for(group, prec, L.geo, g)) return false;
  if (L.nparts) *L.nparts = (int)plq_blocks(g);
  // Non-temporal stores and momentum loads where the two link fields and the
  // momenta exceed the 256 MB Infinity Cache: FP64 32^4 (369 MB) 106.9 against
  // 109.4 us with the stores alone and 124 with neither, FP32 48^4 284.9 /
  // 293.5 / 315; below, FP64 24^4 (117 MB) 43.5 with them and 38.8 without
  const double fields =
      (double)L.geo.nd * L.geo.V * (group == 1 ? 11.0 : 3.0) * (prec == 0 ? 8.0 : 4.0);
  const bool nt = fields > 256.0 * 1024 * 1024;
  if (group == 1 && prec == 0 && L.geo.nd == 4) {
    const size_t nl = 4 * (size_t)L.geo.V;
    const su2_d2 *ia = (const su2_d2 *)L.Uin;
    su2_d2 *oa = (su2_d2 *)L.Uout;
    const QHalf hin{ia, ia + nl};
    const QHalfW hout{oa, oa ? oa + nl : nullptr};
    const quat<double> *rin = (const quat<double> *)L.Uin;
    if (L.in_half) go_wa<PlqSU2<double>, 4>(hin, hout, L, g, nt, st);
    else if (L.out_half) go_wa<PlqSU2<double>, 4>(rin, hout, L, g, nt, st);
    else go_wa<PlqSU2<double>, 4>(rin, (quat<double> *)L.Uout, L, g, nt, st);
    return true;
  }
  if (L.in_half || L.out_half) return false;
#define SU2_PLQ(G, ND)                                                                    \
  go_wa<G, ND>((const typename G::link *)L.Uin, (typename G::link *)L.Uout, L, g, nt, st)
  if (group == 1) {
    if (prec == 0) SU2_PLQ(PlqSU2<double>, 3);
    else if (L.geo.nd == 4) SU2_PLQ(PlqSU2<float>, 4);
    else SU2_PLQ(PlqSU2<float>, 3);
  } else if (L.geo.nd == 4) {
    if (prec == 0) SU2_PLQ(PlqU1<double>, 4);
    else SU2_PLQ(PlqU1<float>, 4);
  } else {
    if (prec == 0) SU2_PLQ(PlqU1<double>, 3);
    else SU2_PLQ(PlqU1<float>, 3);
  }
#undef SU2_PLQ
  return true;
}

}  // namespace su2k
