// su2_sweep.hip -- N_hit Metropolis updates of every link
// (flat_spacetime::sweep, flat-sweep.hh:64-164) for SU(2) and U(1), d = 2, 3, 4.
//
// Order.  The reference walks the even t-slices in parallel and, inside a
// slice, the sites and directions one after another; a GPU needs independent
// links.  The staple of U_mu(x) holds, of the links of direction mu, only
// U_mu(x +- nu) with nu != mu, so for a fixed mu the links of one class of a
// proper colouring of the sites under those neighbour steps are independent.
// Every extent in use even: the two classes of the site parity (sum of the
// coordinates mod 2), 2 nd launches per sweep over V/2 sites each, sites
// computed from the launch index.  Any odd extent: three classes
// c(x) = sum_{nu != mu} h(x_nu) mod 3 with h(k) = k + min(k, a),
// a = (3 - L_nu mod 3) mod 3 (every step along nu changes h by 1 or 2 mod 3,
// the periodic wrap by 1), 3 nd launches over host-built site lists.
//
// One hit (flat-sweep.hh:95-110): R = random_element(delta)
// (random_element.hh:9-25, :27-34), dS = beta/Nc (ReTr(U K) - ReTr(U R K)),
// accept if dS < 0 or v < exp(-dS), then U <- restoreSU(U R); K (the staples,
// get_staples.hh:26-80 with the anisotropy weights) is formed once per link.
//
// Random numbers.  Hit n of link (s, mu) in sweep number w takes one
// Philox4x32-10 block with counter (s nd + mu, n, w_lo, w_hi) and key = seed:
// its words give alpha, u, theta and the acceptance uniform, each as
// (word + 1/2) 2^-32.  The chain therefore depends on (seed, sweep number) only,
// not on the launch shape; it is not the reference's per-thread mt19937 stream.
#include <algorithm>

#include "su2_device.hpp"
#include "su2_launch.hpp"
#include "su2_md_plq.hpp"

using namespace su2dev;

namespace su2k {

constexpr int NTS = 256;

__device__ __forceinline__ double u01_32(uint32_t w) {
  return ((double)w + 0.5) * (1.0 / 4294967296.0);
}

// ReTr(u K) in FP64 (su2.hh:56-58, 72-74; u1.hh:61-67)
__device__ __forceinline__ double retr_mul(const quat<double> &u, const quat<double> &K) {
  return 2.0 * (u.ar * K.ar - u.ai * K.ai - u.br * K.br - u.bi * K.bi);
}
__device__ __forceinline__ double retr_mul_u1(double th, double kre, double kim) {
  double s, c;
  sincos(th, &s, &c);
  return c * kre - s * kim;
}

// sin(pi x) and cos(pi x), |x| < 2^30: r = x - q / 2 exact, |r| <= 1/4, then the
// Taylor series of both in (pi r)^2 <= 0.62 (first terms left out below 2.1e-18)
__device__ __forceinline__ void sincospi_series(double x, double *sn, double *cs) {
  const double q = rint(2.0 * x);
  const double r = M_PI * fma(-0.5, q, x);
  double c, s;
  plq_sincos(r, c, s);
  plq_quadrant((int)q, c, s);
  *sn = s;
  *cs = c;
}

// sqrt(x) for x in [2^-40, 2]: hardware estimate of 1/sqrt and two coupled
// Newton steps (no scaling, no special values)
__device__ __forceinline__ double sqrt_unit(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  double e = fma(-h, g, 0.5);
  g = fma(g, e, g);
  h = fma(h, e, h);
  return fma(fma(-g, g, x), h, g);
}

// v < exp(-dS): decided in FP32 where the two differ by more than 3e-5 of
// their size (the FP32 exponential of an argument up to 100 is good to 1e-5;
// beyond it is below every v > 2^-33), else, and for NaN, by the FP64 function
__device__ __forceinline__ bool below_exp(double v, double dS) {
  const float e = __expf(-(float)dS), w = (float)v;
  if (w < e * (1.0f - 3e-5f)) return true;
  if (w > e * (1.0f + 3e-5f)) return false;
  return v < exp(-dS);
}

// What bounds it: at one hit the link gathers (every second site of a row: half
// of each line a wave touches; a launch of FP64 32^4 fetches 310 to 390 MB from beyond
// the L2, 2.3 to 2.9 times the field, at 6.5 TB/s with one hit and 5.5 with 10),
// beyond a few hits the vector units.  Against blocks dealt round the XCDs,
// one direction at run time, coordinates by division, a branch on the weights
// between the planes' loads and the library's sincospi, sqrt, exp and division: FP64
// 32^4 10 hits 679 -> 520 us, 1 hit 517 -> 411 us, FP32 570 -> 418 and 281 -> 178 us,
// U(1) 24^4 FP64 201 -> 149 us, 8^4 1 hit 65 -> 60 us (before the last two of these:
// FP32 450 and 218, U(1) 153), three colours (15 21 7 32) 168 -> 146 us.
//
// FP64 SU(2), records of 32 bytes: the loads of one plane at a time (all of a side's
// take 128 registers and 20 spills: 619 us) and at most 4 blocks on a CU, held
// by SWEEP_PAD bytes of LDS: with the 7 that the registers allow the blocks' lines
// push each other out of the L2, 550 against 526 us on one card (5 and 3 blocks: 535, 553).  The cap
// was not slower at any size tried (with / without): 16^4 one hit 65.9 / 67.6, 48^4 one hit
// 2176 / 2205, ten 2286 / 2474, d = 3 96^3 188 / 198 and 300 / 304, 128^3 532 / 551, d = 2 2048^2
// 282 / 286, three colours 33^4 741 / 750 us.
constexpr unsigned SWEEP_PAD = 40 * 1024 - 64;
// list == nullptr: the sites of parity `parity` (every extent even);
// otherwise the nlist sites list[0 .. nlist) of one colour class
template <class G, int ND, int mu>
__global__ __launch_bounds__(NTS, 4) void k_sweep(typename G::link *__restrict__ U, Geo geo,
                                               int parity, int tw, const int *__restrict__ list,
                                               int nlist, uint64_t seed, uint64_t sweep,
                                               double delta, int n_hit, double beta_nc,
                                               double w_t, double w_s,
                                               double *__restrict__ partials) {
  using T = typename G::real;
  using link = typename G::link;
  using acc = typename G::acc;
  __shared__ double lds[NTS / 64];
  const int V = geo.V;
  int lb = xcd_block(blockIdx.x, gridDim.x);
  if (tw > 0) {
    const int nb3 = V / 2 / geo.L[0] / NTS, Tc = geo.L[0] / 8;
    const int l = blockIdx.x >> 3, w = l / (tw * nb3), r = l - w * tw * nb3, q = r / tw;
    lb = ((int)(blockIdx.x & 7) * Tc + w * tw + r - q * tw) * nb3 + q;
  }
  const int j = lb * NTS + threadIdx.x;
  double accepted = 0.0;
  if (list ? j < nlist : j < V / 2) {
    int s, up[ND], dn[ND];
    if (list) {
      s = list[j];
      neighbour_offsets<ND>(geo, s, up, dn);
    } else {
      // site j of this parity: pair j of neighbours along the fastest direction
      // (even), and of the two the one with that parity
      int c[ND], rp = 0;
      uint32_t q = 2u * (uint32_t)j;
#pragma unroll
      for (int d = ND - 1; d > 0; --d) {
        const uint32_t Ld = (uint32_t)geo.L[d];
        const uint32_t qn = geo.fdiv ? (geo.mL[d] ? __umulhi(q, geo.mL[d]) : q) : q / Ld;
        c[d] = (int)(q - qn * Ld);
        q = qn;
        if (d < ND - 1) rp += c[d];
      }
      c[0] = (int)q;
      rp += c[0];
      const int odd = (parity + rp) & 1;
      c[ND - 1] += odd;
      s = 2 * j + odd;
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        up[d] = c[d] == geo.L[d] - 1 ? -(geo.L[d] - 1) * geo.str[d] : geo.str[d];
        dn[d] = c[d] == 0 ? (geo.L[d] - 1) * geo.str[d] : -geo.str[d];
      }
    }
    // staples (get_staples.hh:26-80): all upper, then all lower; the weights are 1
    // on an isotropic lattice (a branch round each product would keep the next
    // plane's loads behind it)
    acc K = G::zero();
    link u = U[mu * V + s];
    // one round trip for the links of a side's planes, one for each plane where
    // they are records of 32 bytes
    constexpr bool EACH = sizeof(link) > 16;
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      link l[3 * ND];
      auto fetch = [&](int nu) {
        const int o = side == 0 ? 0 : dn[nu];
        l[3 * nu] = U[nu * V + s + up[mu] + o];
        l[3 * nu + 1] = U[mu * V + s + (side == 0 ? up[nu] : o)];
        l[3 * nu + 2] = U[nu * V + s + o];
      };
      if constexpr (!EACH) {
#pragma unroll
        for (int nu = 0; nu < ND; ++nu)
          if (nu != mu) fetch(nu);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int nu = 0; nu < ND; ++nu) {
        if (nu == mu) continue;
        if (EACH) fetch(nu);
        const acc t = side == 0 ? G::upper(l[3 * nu], l[3 * nu + 1], l[3 * nu + 2])
                                : G::lower(l[3 * nu], l[3 * nu + 1], l[3 * nu + 2]);
        K = G::add(K, G::scale(T((mu == 0 || nu == 0) ? w_t : w_s), t));
        if (EACH) __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    const uint32_t lid = (uint32_t)s * (uint32_t)ND + (uint32_t)mu;
    // ReTr(u K), kept from hit to hit
    [[maybe_unused]] double retr;
    [[maybe_unused]] quat<double> Kd;
    if constexpr (G::NCOMP == 4) {
      Kd = quat<double>{double(K.ar), double(K.ai), double(K.br), double(K.bi)};
      retr = retr_mul(to_d(u), Kd);
    } else {
      retr = retr_mul_u1(double(u), double(K.re), double(K.im));
    }
    for (int n = 0; n < n_hit; ++n) {
      uint32_t c[4] = {lid, (uint32_t)n, (uint32_t)(sweep & 0xffffffffu), (uint32_t)(sweep >> 32)};
      philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
      const double v = u01_32(c[3]);
      if constexpr (G::NCOMP == 4) {
        // random_element (random_element.hh:9-25): (cos a + i sin a u, sin a r (sin th + i cos th))
        // alpha = 2 pi delta u0 and theta = 2 pi u2 through sincospi (no
        // argument reduction by pi)
        const double uu = -1.0 + 2.0 * u01_32(c[1]);
        const double r = sqrt_unit(1.0 - uu * uu);
        double sa, ca, st, ct;
        double x = 2.0 * delta * u01_32(c[0]);
        if (fabs(delta) > 1e6) x = fma(-2.0, rint(0.5 * x), x);  // a whole number of turns off
        sincospi_series(x, &sa, &ca);
        sincospi_series(2.0 * u01_32(c[2]), &st, &ct);
        const quat<double> R{ca, sa * uu, sa * r * st, sa * r * ct};
        const quat<double> ud = to_d(u);
        const quat<double> uR = qmul(ud, R);
        const double dS = beta_nc * (retr - retr_mul(uR, Kd));
        if (dS < 0.0 || below_exp(v, dS)) {
          // restoreSU (su2.hh:62-66) in FP64, one rounding to the storage precision;
          // 1/sqrt(1 + d) = 1 - d/2 + 3 d^2/8 - ... (5 d^3/16 < 4e-17 below 5e-6)
          const double d = fma(uR.ar, uR.ar, fma(uR.ai, uR.ai, fma(uR.br, uR.br, fma(uR.bi, uR.bi, -1.0))));
          const double rn = fabs(d) < 5e-6 ? fma(d, fma(0.375, d, -0.5), 1.0) : 1.0 / sqrt(1.0 + d);
          u = link{T(uR.ar * rn), T(uR.ai * rn), T(uR.br * rn), T(uR.bi * rn)};
          retr = retr_mul(to_d(u), Kd);
          accepted += 1.0;
        }
      } else {
        // random_element (random_element.hh:27-34): phase in [-pi delta, pi delta)
        const double th = -M_PI * delta + (2.0 * M_PI * delta) * u01_32(c[0]);
        const double ud = double(u), un = ud + th;
        const double rn = retr_mul_u1(un, double(K.re), double(K.im));
        const double dS = beta_nc * (retr - rn);
        if (dS < 0.0 || below_exp(v, dS)) {
          u = T(un);
          retr = sizeof(T) == 8 ? rn : retr_mul_u1(double(u), double(K.re), double(K.im));
          accepted += 1.0;
        }
      }
    }
    U[mu * V + s] = u;
  }
  const double r = block_sum<NTS>(accepted, lds);
  if (threadIdx.x == 0) partials[lb] = r;
}

// The order of the blocks.  Each XCD walks one contiguous eighth of the sites.  Where
// the t slices divide into eighths and into blocks (tw > 0), it walks them in groups of
// tw slices, t fastest within a group, so that a block's t neighbours were fetched by
// the blocks just before it into the same L2.  Groups of 4 to 7 slices: slices lie a
// whole number of L2 ways apart where the extents are powers of two, and then eight or
// more of them push each other out (FP64, one hit, groups of 4 / 8 / all slices / memory
// order: 128^3 d = 3 415 / 486 / 530 / 430 us, 32^3 x 128 1667 / 1911 / 2081 / 1872, 64^4 6786 /
// 7453 / 7453 / 7834); elsewhere longer groups are as good (40^4 in 5 1043, memory order
// 1189; 48^4 in 6 2176, in 3 2206, memory order 2433 us).
static int sweep_tw(const Geo &g) {
  if (g.L[0] % 8 != 0 || (g.V / 2 / g.L[0]) % NTS != 0) return 0;
  const int Tc = g.L[0] / 8;
  int tw = std::min(Tc, 7);
  while (Tc % tw != 0) --tw;
  return tw;
}

int sweep_blocks(const Geo &g, int nlist) { return ((nlist >= 0 ? nlist : g.V / 2) + NTS - 1) / NTS; }

template <class G, int ND>
static void sweep_nd(void *U, const Geo &g, int mu, int parity, const int *list, int nlist,
                     uint64_t seed, uint64_t sweep, double delta, int n_hit, double beta_nc,
                     double w_t, double w_s, double *partials, hipStream_t st) {
  using link = typename G::link;
  const dim3 grid(sweep_blocks(g, list ? nlist : -1));
  if (grid.x == 0) return;
#define SU2_SWEEP(M)                                                                          \
  hipLaunchKernelGGL((k_sweep<G, ND, M>), grid, dim3(NTS), sizeof(link) > 16 ? SWEEP_PAD : 0, st, (link *)U,    \
                     g, parity, list ? 0 : sweep_tw(g), list, nlist, seed, sweep, delta, n_hit, beta_nc, w_t, w_s, partials)
  if (mu == 0) SU2_SWEEP(0);
  else if (mu == 1) SU2_SWEEP(1);
  else if (ND > 2 && mu == 2) SU2_SWEEP((ND > 2 ? 2 : 0));
  else SU2_SWEEP((ND > 3 ? 3 : 0));
#undef SU2_SWEEP
}

void launch_sweep(int group, int prec, void *U, const Geo &g, int mu, int parity, const int *list,
                  int nlist, uint64_t seed, uint64_t sweep, double delta, int n_hit,
                  double beta_nc, double w_t, double w_s, double *partials,
                  hipStream_t st) {
#define SWEEP_ARGS U, g, mu, parity, list, nlist, seed, sweep, delta, n_hit, beta_nc, w_t, w_s, partials, st
#define SWEEP_G(G)                               \
  do {                                           \
    if (g.nd == 2) sweep_nd<G, 2>(SWEEP_ARGS);   \
    else if (g.nd == 3) sweep_nd<G, 3>(SWEEP_ARGS); \
    else sweep_nd<G, 4>(SWEEP_ARGS);             \
  } while (0)
  if (group == 1) {
    if (prec == 0) SWEEP_G(GSU2<double>);
    else SWEEP_G(GSU2<float>);
  } else {
    if (prec == 0) SWEEP_G(GU1<double>);
    else SWEEP_G(GU1<float>);
  }
#undef SWEEP_G
#undef SWEEP_ARGS
}

}  // namespace su2k
