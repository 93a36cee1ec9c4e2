// su2_clover.hip -- plaquette sums, clover energy density and topological charge
// of an SU(2) lattice in d = 4 in one pass (retr_sum_Wplaquettes,
// flat-gauge_energy.hpp:31-94; energy_density, flat-energy_density.hh:57-164).
//
// The clover of a plane at x is the sum of the four plaquettes that touch x, each
// read from x on.  A plaquette P = a b c^+ d^+ of the site y (a = U_mu(y), b =
// U_nu(y+mu), c = U_mu(y+nu), d = U_nu(y)) therefore serves four sites: with
// M = a b and N = d c its imaginary part is
//   at y       Im(M N^+)          at y+mu     Im(b N^+ a)
//   at y+nu    Im(d^+ M c^+)      at y+mu+nu  Im(N^+ M)
// It is evaluated once, by the layout of su2_md_plq.hpp: the terms of y+t stay in
// registers, those along the two fastest directions go through LDS, those from
// x-1 are evaluated twice, and a row whose row below is in another block
// evaluates that row's terms itself.  A term for a later slice (t and a second
// direction) waits with its sender and goes out with the next slice's.
//
// One thread per site and four leaves of three products per plane (the kernel
// of the other groups and dimensions) takes 192 against 112 multiply-adds per
// plane and some 56 against 13 link loads per site, and is bound by those loads.
// This one is bound by its two round trips per slice (2 waves per SIMD, 256
// registers).  energy_density with its reduction and synchronisation, before and
// now: FP64 48^4 762 -> 466 us, 32^4 164 -> 100, 24^4 63 -> 50, FP32 32^4 107 -> 77, 48^4
// 457 -> 354 us; the plaquette sums that the flow table takes beside it (two
// kernels of 11 us at 24^4) and its second clover pass (35 us) come for free.
#include "su2_md_plq.hpp"

namespace su2k {

namespace {

constexpr int CUS = 256;

// LDS: the links per thread and of a halo row, seven terms per thread
template <typename T> constexpr int clv_lrec() { return PlqSU2<T>::lrec(4); }
constexpr int CLV_VREC = (7 * 3 | 1) * 8;
template <typename T> size_t clv_lds(const PlqGeo &g) {
  const size_t nt = plq_threads(g);
  return (nt + g.L[3]) * clv_lrec<T>() + nt * CLV_VREC;
}

struct CluTerms {
  pv3<double> v0, vb, vc, vd;  // at y, y+mu, y+nu, y+mu+nu
};
template <int WANT>  // bits: 1 v0, 2 vb, 4 vc, 8 vd
__device__ __forceinline__ void clv_plane(const quat<double> &a, const quat<double> &b,
                                          const quat<double> &c, const quat<double> &d,
                                          CluTerms &o, double *re = nullptr) {
  const quat<double> M = qmul_fma(a, b), N = qmul_fma(d, c);
  if (WANT & 1) o.v0 = qim(M, qdag(N));
  if (re) *re += qre(M, qdag(N));
  if (WANT & 2) o.vb = qim(b, qmul_fma(qdag(N), a));
  if (WANT & 4) o.vc = qim(qmul_fma(qdag(d), M), qdag(c));
  if (WANT & 8) o.vd = qim(qdag(N), M);
}
__device__ __forceinline__ void vacc(double (&g)[3], const pv3<double> &v) {
#pragma unroll
  for (int k = 0; k < 3; ++k) g[k] += v.k[k];
}
__device__ __forceinline__ pv3<double> vsum(const pv3<double> &u, const pv3<double> &v) {
  return pv3<double>{{u.k[0] + v.k[0], u.k[1] + v.k[1], u.k[2] + v.k[2]}};
}
__device__ __forceinline__ double vdot(const double (&u)[3], const double (&v)[3]) {
  return fma(u[0], v[0], fma(u[1], v[1], u[2] * v[2]));
}

// partials rows: 0 / 1 the temporal / spatial plaquettes' ReTr, 2 / 3 the
// temporal / spatial planes' ReTr(G G), 4 the charge density's sum
template <typename T>
__global__ __launch_bounds__(PLQ_NT, 2) void k_clover_plq(const quat<T> *__restrict__ Uin, PlqGeo g,
                                                        double *__restrict__ partials,
                                                        int pstride) {
  extern __shared__ __align__(16) char smem[];
  const int nt = (int)blockDim.x, tid = (int)threadIdx.x;
  const PlqSite f = plq_site(g, blockIdx.x, gridDim.x, (uint32_t)tid, (uint32_t)nt);
  const size_t V = (size_t)g.V;
  constexpr int LREC = clv_lrec<T>();
  char *const lv0 = smem + (nt + g.L[3]) * LREC;
  char *const lown = smem + tid * LREC, *const lrow = smem + f.lur * LREC,
             *const lz0 = smem + f.luz * LREC;
  char *const vown = lv0 + tid * CLV_VREC, *const vrow = lv0 + f.ldr * CLV_VREC,
             *const vz = lv0 + f.ldz * CLV_VREC;
  const quat<T> *U[4];
#pragma unroll
  for (int m = 0; m < 4; ++m) U[m] = Uin + (size_t)m * V;
  const bool rin = f.rin, din = f.ldr >= 0;
  char *const vdiag = lv0 + (din && f.active ? f.ldr + f.dz : tid) * CLV_VREC;
  const bool edge = __builtin_amdgcn_readfirstlane((int)(__ballot(!din) != 0)) != 0;
  auto ld = [&](int m, int i) { return ldq(U[m], (uint32_t)i); };
  auto D = [](const quat<T> &q) { return to_d(q); };

  double sums[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  quat<T> own[4], xl;
  // what the slice below left: the y+t terms of the planes (t, i) at this site,
  // the y+t+x term of (t, x) at x-1, the y+t+r and y+t+z terms to send on, and for
  // an edge row the y+t+r term of the row below
  pv3<double> cb[4], cdx, cvr, cvz, ce{};
  int s = f.t0 * g.vol3 + f.o3;
  {
    const int dt = f.t0 == 0 ? (g.L[0] - 1) * g.vol3 : -g.vol3;
    CluTerms o;
    const quat<T> a = ld(0, s + dt);
    const int up[4] = {0, f.ux, f.ur, f.uz};
#pragma unroll
    for (int i = 1; i < 4; ++i) {
      own[i] = ld(i, s);
      const quat<T> c = ld(0, s + dt + up[i]), d = ld(i, s + dt);
      if (i == 1) clv_plane<2>(D(a), D(own[i]), D(c), D(d), o);
      else clv_plane<10>(D(a), D(own[i]), D(c), D(d), o);
      cb[i] = o.vb;
      if (i == 2) cvr = o.vd;
      if (i == 3) cvz = o.vd;
    }
    xl = ld(1, s + f.dx);
    clv_plane<8>(D(ld(0, s + dt + f.dx)), D(xl), D(a), D(ld(1, s + dt + f.dx)), o);
    cdx = o.vd;
    if (!din) {
      clv_plane<8>(D(ld(0, s + dt + f.dr)), D(ld(2, s + f.dr)), D(a), D(ld(2, s + dt + f.dr)), o);
      ce = o.vd;
    }
  }
  for (int t = f.t0; t < f.t1; ++t) {
    const int ut = t == g.L[0] - 1 ? -(g.L[0] - 1) * g.vol3 : g.vol3;
    double G[6][3];  // planes tx, tr, tz, xr, xz, rz
    quat<T> nx[4], ux[4], xlt;
    pv3<double> lr, lz;  // y+x+r, y+x+z terms of the planes (x, r), (x, z) at x-1
    {
      quat<T> lx[4], lxu[4];
      own[0] = ld(0, s);
      lx[0] = ld(0, s + f.dx);
      xlt = ld(1, s + f.dx + ut);
      lx[2] = ld(2, s + f.dx);
      lxu[2] = ld(1, s + f.dx + f.ur);
      lx[3] = ld(3, s + f.dx);
      lxu[3] = ld(1, s + f.dx + f.uz);
      if (!rin) {
        quat<T> h[3] = {ld(0, s + f.ur), ld(1, s + f.ur), ld(3, s + f.ur)};
        plq_put(lrow, 0, h[0]);
        plq_put(lrow, 1, h[1]);
        plq_put(lrow, 3, h[2]);
      }
#pragma unroll
      for (int i = 1; i < 4; ++i) nx[i] = ld(i, s + ut);
      ux[2] = ld(2, s + f.ux);
      ux[3] = ld(3, s + f.ux);
      ux[0] = ld(0, s + f.ux);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < 4; ++m) plq_put(lown, m, own[m]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int p = 0; p < 6; ++p) G[p][0] = G[p][1] = G[p][2] = 0.0;
      vacc(G[0], cb[1]);
      vacc(G[1], cb[2]);
      vacc(G[2], cb[3]);
      vacc(G[0], cdx);
      CluTerms o;
      clv_plane<12>(D(lx[0]), D(xlt), D(own[0]), D(xl), o);
      vacc(G[0], o.vc);
      cdx = o.vd;
      clv_plane<10>(D(xl), D(own[2]), D(lxu[2]), D(lx[2]), o);
      vacc(G[3], o.vb);
      lr = o.vd;
      clv_plane<10>(D(xl), D(own[3]), D(lxu[3]), D(lx[3]), o);
      vacc(G[4], o.vb);
      lz = o.vd;
      plq_pin(cdx.k);
      plq_pin(lr.k);
      plq_pin(lz.k);
#pragma unroll
      for (int p = 0; p < 6; ++p) plq_pin(G[p]);
      __builtin_amdgcn_sched_barrier(0);
    }
    plq_barrier();
    {
      CluTerms o;
      double rt = 0.0, rs = 0.0;
      quat<T> p, q;
      auto put = [&](int k, const pv3<double> &v) { plq_putv<PlqSU2<double>>(vown, k, v); };
      // (r, z): y+r, y+z, y+r+z terms
      plq_get(lrow, 3, p);
      plq_get(lz0, 2, q);
      clv_plane<15>(D(own[2]), D(p), D(q), D(own[3]), o, &rs);
      vacc(G[5], o.v0);
      put(2, o.vb);
      put(5, o.vc);
      put(6, o.vd);
      __builtin_amdgcn_sched_barrier(0);
      // (t, r), (t, z): the y+r (y+z) term, with the slice below's y+t+r (y+t+z) one
      plq_get(lrow, 0, p);
      clv_plane<15>(D(own[0]), D(nx[2]), D(p), D(own[2]), o, &rt);
      vacc(G[1], o.v0);
      put(0, vsum(o.vc, cvr));
      cb[2] = o.vb;
      cvr = o.vd;
      __builtin_amdgcn_sched_barrier(0);
      plq_get(lz0, 0, q);
      clv_plane<15>(D(own[0]), D(nx[3]), D(q), D(own[3]), o, &rt);
      vacc(G[2], o.v0);
      put(3, vsum(o.vc, cvz));
      cb[3] = o.vb;
      cvz = o.vd;
      __builtin_amdgcn_sched_barrier(0);
      // (x, r), (x, z): the y+r (y+z) term, with x-1's y+x+r (y+x+z) one
      plq_get(lrow, 1, p);
      clv_plane<5>(D(own[1]), D(ux[2]), D(p), D(own[2]), o, &rs);
      vacc(G[3], o.v0);
      put(1, vsum(o.vc, lr));
      __builtin_amdgcn_sched_barrier(0);
      plq_get(lz0, 1, q);
      clv_plane<5>(D(own[1]), D(ux[3]), D(q), D(own[3]), o, &rs);
      vacc(G[4], o.v0);
      put(4, vsum(o.vc, lz));
      __builtin_amdgcn_sched_barrier(0);
      clv_plane<3>(D(own[0]), D(nx[1]), D(ux[0]), D(own[1]), o, &rt);
      vacc(G[0], o.v0);
      cb[1] = o.vb;
      if (f.active) {
        sums[0] += 2.0 * rt;
        sums[1] += 2.0 * rs;
      }
      plq_pin(sums);
#pragma unroll
      for (int k = 0; k < 6; ++k) plq_pin(G[k]);
#pragma unroll
      for (int i = 1; i < 4; ++i) plq_pin(cb[i].k);
      plq_pin(cvr.k);
      plq_pin(cvz.k);
      __builtin_amdgcn_sched_barrier(0);
      if (edge) {
        // the row below is in another block: its terms, for the lanes of that row
        const int y = s + f.dr;
        const quat<T> eR = ld(2, y), e0 = ld(0, y), eRt = ld(2, y + ut), eX = ld(1, y),
                      eRx = ld(2, y + f.ux);
        const double w = din ? 0.0 : 1.0;
        auto wacc = [&](double (&gg)[3], const pv3<double> &v) {
#pragma unroll
          for (int k = 0; k < 3; ++k) gg[k] = fma(w, v.k[k], gg[k]);
        };
        clv_plane<12>(D(e0), D(eRt), D(own[0]), D(eR), o);
        wacc(G[1], o.vc);
        wacc(G[1], ce);
        ce = o.vd;
        clv_plane<4>(D(eX), D(eRx), D(own[1]), D(eR), o);
        wacc(G[3], o.vc);
        plq_pin(G[1]);
        plq_pin(G[3]);
        plq_pin(ce.k);
        __builtin_amdgcn_sched_barrier(0);
        // in two round trips: all twelve links at once do not fit the registers
        const quat<T> eX1 = ld(1, y + f.dx), eR1 = ld(2, y + f.dx), eRz = ld(2, y + f.uz),
                      eZ = ld(3, y), eR2 = ld(2, y + f.dz), eZ2 = ld(3, y + f.dz),
                      zZ = ld(3, s + f.dz);
        clv_plane<8>(D(eX1), D(eR), D(xl), D(eR1), o);
        wacc(G[3], o.vd);
        clv_plane<2>(D(eR), D(own[3]), D(eRz), D(eZ), o);
        wacc(G[5], o.vb);
        clv_plane<8>(D(eR2), D(zZ), D(eR), D(eZ2), o);
        wacc(G[5], o.vd);
      }
    }
    plq_barrier();
    {
      pv3<double> v;
      auto get = [&](const char *rec, int k, double (&gg)[3]) {
        plq_getv<PlqSU2<double>>(rec, k, v);
        vacc(gg, v);
      };
      get(vz, 3, G[2]);
      get(vz, 4, G[4]);
      get(vz, 5, G[5]);
      if (din) {
        get(vrow, 0, G[1]);
        get(vrow, 1, G[3]);
        get(vrow, 2, G[5]);
        get(vdiag, 6, G[5]);
      }
      if (f.active) {
        sums[2] -= 2.0 * (vdot(G[0], G[0]) + vdot(G[1], G[1]) + vdot(G[2], G[2]));
        sums[3] -= 2.0 * (vdot(G[3], G[3]) + vdot(G[4], G[4]) + vdot(G[5], G[5]));
        sums[4] -= 4.0 * ((vdot(G[0], G[5]) - vdot(G[1], G[4])) + vdot(G[2], G[3]));
      }
      plq_pin(sums);
#pragma unroll
      for (int i = 1; i < 4; ++i) own[i] = nx[i];
      xl = xlt;
      s += ut;
    }
  }
  __syncthreads();
  double *l5 = (double *)smem;
  const int lane = tid & 63, wv = tid >> 6, nw = nt >> 6;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    double v = sums[k];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if (lane == 0) l5[k * 4 + wv] = v;
  }
  __syncthreads();
  if (tid < 5) {
    double v = 0.0;
    for (int i = 0; i < nw; ++i) v += l5[tid * 4 + i];
    partials[(size_t)tid * pstride + blockIdx.x] = v;
  }
}

// Not where more than half of the lanes of many blocks hold no site (planes y z of
// few sites; this / the kernel of the other groups, energy_density in FP64, x y z t):
// 64 5 5 64 33.9 / 31.9, 64 3 3 64 34.4 / 27.6, 128 1 2 256 95 / 27.6 us; 64 6 6 64 34.0 / 35.8 us;
// up to 131072 lanes the launches count: 32 5 5 32 24.0 / 27.4, 32 1 2 32 23.6 / 25.3, 32 4 4
// 64 27.2 / 27.0 us.
template <typename T> bool clv_geo(const Geo &geo, PlqGeo &g) {
  // FP64: three waves per block, so that two blocks' LDS fits a CU
  const int threads = sizeof(T) == 8 ? 192 : PLQ_NT;
  if (geo.nd != 4 || !make_plq_rows(geo.L, 4, geo.V, g, threads) || !plq_full(g)) return false;
  const int waves = (int)plq_threads(g) / 64;
  const int percu = std::max(1, std::min(8 / waves, (int)(160 * 1024 / clv_lds<T>(g))));
  return make_plq_chunks(percu, CUS, g);
}

}  // namespace

int clover_partials(int group, int prec, const Geo &geo) {
  PlqGeo g;
  if (group != 1 || !(prec == 0 ? clv_geo<double>(geo, g) : clv_geo<float>(geo, g))) return 0;
  return (int)plq_blocks(g);
}

int launch_clover(int group, int prec, const void *U, const Geo &geo, double *partials, int pstride,
                  hipStream_t st) {
  PlqGeo g;
  if (group != 1 || !(prec == 0 ? clv_geo<double>(geo, g) : clv_geo<float>(geo, g))) return 0;
  const dim3 grid(plq_blocks(g)), block(plq_threads(g));
  if (prec == 0)
    hipLaunchKernelGGL((k_clover_plq<double>), grid, block, (unsigned)clv_lds<double>(g), st,
                       (const quat<double> *)U, g, partials, pstride);
  else
    hipLaunchKernelGGL((k_clover_plq<float>), grid, block, (unsigned)clv_lds<float>(g), st,
                       (const quat<float> *)U, g, partials, pstride);
  return (int)plq_blocks(g);
}

}  // namespace su2k
