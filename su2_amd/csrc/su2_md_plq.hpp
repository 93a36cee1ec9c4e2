// su2_md_plq.hpp -- the fused force / momentum / link update from shared
// plaquettes (get_staples.hh:26-80, flat-gaugemonomial.hh:105-131,
// update_momenta.hh:27-30, update_gauge.hh:11-14), SU(2) and U(1), d = 3, 4.
//
// The force of a link is a sum over its plaquettes, and a plaquette
// P = a b c^+ d^+ (a = U_mu(x), b = U_nu(x+mu), c = U_mu(x+nu), d = U_nu(x))
// serves four links:
//   Im(U K):  a: +Im(P)            b: Im(b c^+ d^+ a)
//             d: -Im(P)            c: Im(c b^+ a^+ d)
// With M = a b and N = d c: P = M N^+, b c^+ d^+ a = b (N^+ a) and
// c b^+ a^+ d = c (M^+ d).  A thread takes the site x, evaluates its planes
// once and hands the b and c terms on to the sites x+mu and x+nu, where the
// staple form evaluates every plaquette four times and loads 18 neighbour
// links per link (10.75 with the links carried along t).  Here:
//   * t: a thread walks the slices of a t-chunk upwards; the b terms of its
//     planes (t, i) belong to its own next links and stay in registers, as do
//     the links U_i(x+t) and U_1(x-1+t);
//   * the two fastest directions: a block holds whole rows of the fastest one
//     at one x (d = 4), links and terms are exchanged through LDS; a row whose
//     neighbour row is in another block loads that row's links, and evaluates
//     the terms it would have been handed itself;
//   * x (d = 4): never in the block; the terms from x-1 are always evaluated
//     here (three half planes, a quarter of the arithmetic).
// d = 4: 13 link loads per site (3.25 per link) plus the edge rows'.
//
// Two barriers per slice; they wait for LDS only (asm, lgkmcnt), so global
// loads stay in flight across them.
//
// What bounds it, and what it measured (steps with HIP events, against the
// t-walk of the staple form, same box).  The staple form is bound by its link
// requests (31 vector memory instructions per 64 links); this one has 15 and is
// bound by the bytes beyond the L2 and the latency of two round trips per slice
// (links; momenta and edge-row links, which are loaded together while the last
// planes are evaluated).  FP64: 32^4 143 -> 107 us (565 MB beyond the L2, 5.3
// TB/s), 48^4 784 -> 518 us (112 B per link at 4.6 TB/s), 40^4 386 -> 287 us,
// 24^4 48.6 -> 38.9 us, momentum-only 32^4 115 -> 82 us.  FP32: 48^4 384 -> 277
// us, 40^4 188 -> 150 us, 28^4 45.5 -> 41.0 us, 32^4 a tie (55.5 to 61.6 / 58.2 to 61.4
// us over four cards).  U(1), where the
// staple form takes seven sine / cosine pairs per link and this one six sines per
// site and three for x-1: FP64 24^4 33.8 -> 18.9 us (16.4 in a trace, without the events), 32^4 85.5 -> 38.0 us, d = 3
// 64^3 17.8 -> 11.0 us; FP32 32^4 46.7 -> 24.6 us.  Loading the
// next slice's first links during the update spills (FP64) and makes the next
// slice wait for the update's stores, which share the counter of the loads:
// 137 us at 32^4.
#pragma once
#include <algorithm>
#include <cmath>

#include "su2_md_fast.hpp"

namespace su2k {

// ------------------------------------------------------------------ layout --
constexpr int PLQ_NT = 256;            // most threads of a block
constexpr int PLQ_ROW = 128;           // longest row

struct PlqGeo {
  int L[4];      // extents t, x, y, z (1 above nd)
  int str[4];    // site strides
  int V, nd;
  int vol3;      // sites of a t slice
  int rpb;       // rows (of the fastest direction) per block
  int nrows;     // rows per x plane (d = 4) or per slice (d = 3)
  int nyb;       // blocks per x plane: ceil(nrows / rpb)
  int nb3;       // blocks per slice
  int Tc, nchunk;
  uint32_t mLf;  // multiply-high divisors (fast_div): fastest extent, nyb, nb3
  uint32_t mnyb, mnb3;
};

// (chunk, block) pair lb, thread tid -> site of the slice, chunk, row and neighbours
struct PlqSite {
  bool active;
  int o3;              // site within the slice
  int t0, t1;          // slices [t0, t1)
  int ux, dx;          // +-x neighbour offsets (d = 4)
  int ur, dr;          // +- row direction
  int uz, dz;          // +- fastest direction
  bool rin;            // the row above is in this block
  int lur, ldr;        // the row neighbours' thread; the halo's slot, -1 where in another block
  int luz, ldz;        // the fastest direction's neighbours' thread
};
__host__ __device__ __forceinline__ PlqSite plq_site_at(const PlqGeo &g, uint32_t lb, uint32_t tid,
                                                        uint32_t nt) {
  PlqSite f;
  const uint32_t chunk = fast_div(lb, g.mnb3);
  const uint32_t b3 = lb - chunk * (uint32_t)g.nb3;
  f.t0 = (int)chunk * g.Tc;
  f.t1 = f.t0 + g.Tc < g.L[0] ? f.t0 + g.Tc : g.L[0];
  const uint32_t x = fast_div(b3, g.mnyb);
  const int r0 = (int)(b3 - x * (uint32_t)g.nyb) * g.rpb;
  const int Lf = g.L[g.nd - 1], Lr = g.nrows;
  const int nr = Lr - r0 < g.rpb ? Lr - r0 : g.rpb;  // rows of this block
  const uint32_t row = fast_div(tid, g.mLf);
  const int z = (int)(tid - row * (uint32_t)Lf);
  f.active = (int)row < nr;
  const int r = f.active ? (int)row : 0;
  const int y = r0 + r;
  f.o3 = (int)x * (Lr * Lf) + y * Lf + z;
  const int plane = Lr * Lf;
  f.ux = ((int)x == g.L[1] - 1) ? -(g.L[1] - 1) * plane : plane;
  f.dx = (x == 0) ? (g.L[1] - 1) * plane : -plane;
  const int yu = (y == Lr - 1) ? 0 : y + 1, yd = (y == 0) ? Lr - 1 : y - 1;
  f.ur = (yu - y) * Lf;
  f.dr = (yd - y) * Lf;
  f.uz = (z == Lf - 1) ? -(Lf - 1) : 1;
  f.dz = (z == 0) ? Lf - 1 : -1;
  f.rin = yu >= r0 && yu < r0 + nr;
  f.lur = f.rin ? (int)tid + f.ur : (int)nt + z;
  f.ldr = (yd >= r0 && yd < r0 + nr) ? (int)tid + f.dr : -1;
  f.luz = (int)tid + f.uz;
  f.ldz = (int)tid + f.dz;
  if (!f.active) {
    // a lane past the block's rows: reads as its first row's lane z, exchanges
    // with itself, writes nothing
    f.rin = true;
    f.lur = f.ldr = f.luz = f.ldz = (int)tid;
  }
  return f;
}
// the same where each XCD walks one contiguous eighth of the (chunk, block) sequence
__host__ __device__ __forceinline__ PlqSite plq_site(const PlqGeo &g, uint32_t b, uint32_t nblk,
                                                     uint32_t tid, uint32_t nt) {
  const uint32_t xcd = b & 7u, local = b >> 3, per = nblk >> 3, rem = nblk & 7u;
  return plq_site_at(g, xcd * per + (xcd < rem ? xcd : rem) + local, tid, nt);
}

inline uint32_t plq_blocks(const PlqGeo &g) { return (uint32_t)g.nb3 * (uint32_t)g.nchunk; }
__host__ __device__ inline uint32_t plq_threads(const PlqGeo &g) {
  return (uint32_t)((g.rpb * g.L[g.nd - 1] + 63) / 64 * 64);
}

// The rows of a block for extents L (t, x, y, z; nd = 3, 4); false where the
// step does not apply.  rpb: the rows that waste the fewest lanes of at most
// `threads`, fewer edge rows breaking ties.
inline bool make_plq_rows(const int L[4], int nd, int V, PlqGeo &g, int threads = PLQ_NT) {
  if (nd < 3 || nd > 4) return false;
  for (int k = 0; k < 4; ++k) g.L[k] = L[k];
  g.nd = nd;
  g.V = V;
  g.str[3] = 1;
  g.str[2] = L[3];
  g.str[1] = L[2] * L[3];
  g.str[0] = L[1] * L[2] * L[3];
  g.vol3 = g.str[0];
  const int Lf = L[nd - 1];
  g.nrows = L[nd - 2];
  if (Lf > PLQ_ROW || Lf < 2) return false;
  const uint64_t two32 = 1ull << 32;
  if ((uint64_t)V * 32u >= two32) return false;  // 32-bit byte offsets in a plane
  double best = 0.0;
  g.rpb = 0;
  for (int r = 1; r <= g.nrows && r * Lf <= threads; ++r) {
    const int nyb = (g.nrows + r - 1) / r, nt = (r * Lf + 63) / 64 * 64;
    // useful rows per lane, less the edge rows' terms (a fifth of a row each,
    // none where the block holds every row)
    const double eff = (double)g.nrows * Lf / ((double)nyb * nt) /
                       (1.0 + (nyb > 1 ? 0.2 / r : 0.0));
    if (eff > best * 1.0001) {
      best = eff;
      g.rpb = r;
    }
  }
  if (g.rpb < 1) return false;
  g.nyb = (g.nrows + g.rpb - 1) / g.rpb;
  g.nb3 = g.nyb * (nd == 4 ? L[1] : 1);
  g.mLf = fast_div_magic((uint32_t)Lf);
  return true;
}

// share of the lanes that hold a site
inline double plq_fill(const PlqGeo &g) {
  return (double)g.nrows * g.L[g.nd - 1] / ((double)g.nyb * plq_threads(g));
}

// lanes mostly in use, or a launch so small that idle ones do not show (measured where
// it is used)
inline bool plq_full(const PlqGeo &g) {
  return plq_fill(g) >= 0.5 || (double)g.nb3 * plq_threads(g) * g.L[0] <= 131072.0;
}

// The t-chunks where `percu` blocks are resident on each of `cus` CUs.  A slice
// of a resident round costs a latency and a share per resident wave, in the
// ratio 2 : 1 (FP32 32^4, measured: chunks of 8 slices, 8 waves per CU, 58.5 us;
// of 6, 12 waves, 60.8; of 4, two rounds, 60.3; FP64 24^4: 4 slices 39, 3 slices
// 43.7, 2 slices 43.2 us), a chunk's first slice a third more (the terms of
// the slice below it).
inline bool make_plq_chunks(int percu, int cus, PlqGeo &g) {
  const int waves = (g.rpb * g.L[g.nd - 1] + 63) / 64;
  const long round = (long)percu * cus;
  double cost = 1e300;
  g.Tc = 1;
  for (int Tc = 1; Tc <= g.L[0]; ++Tc) {
    const long nb = (long)g.nb3 * ((g.L[0] + Tc - 1) / Tc), full = (nb - 1) / round;
    const long last = (nb - full * round + cus - 1) / cus;
    const double c =
        (Tc + 0.35) * ((double)full * (2.0 + percu * waves) + 2.0 + (double)(last * waves));
    if (c < cost * 0.999) {
      cost = c;
      g.Tc = Tc;
    }
    if (nb <= cus) break;  // one block on some of the CUs: longer chunks only cost more
  }
  g.nchunk = (g.L[0] + g.Tc - 1) / g.Tc;
  if ((uint64_t)g.nb3 * g.nchunk * g.nb3 >= (1ull << 32)) return false;
  g.mnyb = fast_div_magic((uint32_t)g.nyb);
  g.mnb3 = fast_div_magic((uint32_t)g.nb3);
  return true;
}

// ------------------------------------------------------------ the algebra --
template <typename T> struct pv3 {
  T k[3];
};
template <typename T> struct pv4 {
  T k[4];  // Re a, Im a, Re b, Im b
};

// acc += w v
template <int N, typename V>
__device__ __forceinline__ void plq_add(double (&acc)[N], double w, const V &v) {
#pragma unroll
  for (int k = 0; k < N; ++k) acc[k] = fma(w, double(v.k[k]), acc[k]);
}

// Im(u v) in momentum order (bi, br, ai)
template <typename T> __device__ __forceinline__ pv3<T> qim(const quat<T> &u, const quat<T> &v) {
  pv3<T> r;
  r.k[2] = fma(u.ar, v.ai, fma(u.ai, v.ar, fma(-u.bi, v.br, u.br * v.bi)));
  r.k[1] = fma(u.ar, v.br, fma(-u.ai, v.bi, fma(u.br, v.ar, u.bi * v.ai)));
  r.k[0] = fma(u.ar, v.bi, fma(u.ai, v.br, fma(u.bi, v.ar, -(u.br * v.ai))));
  return r;
}
template <typename T> __device__ __forceinline__ double qre(const quat<T> &u, const quat<T> &v) {
  return double(fma(u.ar, v.ar, -fma(u.ai, v.ai, fma(u.br, v.br, u.bi * v.bi))));
}

// SU(2).  NM: reals of a momentum, NV: of a plaquette's term of a link.
// FP64: a term is Im(U K) of that plaquette, three reals; the b and a terms of a
// plaquette's links are theirs, a and d share theirs but for the sign.
template <typename T_> struct PlqSU2 {
  using T = T_;
  using link = quat<T>;
  static constexpr int NM = 3, NV = 3;
  using V = pv3<T>;
  // P' = P - DF coef ep Im(U K); a plaquette adds RP re to the sum of ReTr(U K) over its links
  static constexpr double DF = 2.0, RP = 8.0;
  // LDS bytes of ND links, an odd multiple of 16
  static constexpr int lrec(int nd) { return (nd * (int)sizeof(link) / 16 | 1) * 16; }
  // the terms of a and d into their sums, those of b and c out; B, C: whether the b /
  // c term is wanted; RE: re += ReTr(P) / 2
  template <bool B, bool C, bool RE>
  __device__ static void plane(const link &a, const link &b, const link &c, const link &d,
                               double (&sa)[NV], double (&sd)[NV], V &vb, V &vc, double w,
                               double &re) {
    const link M = qmul_fma(a, b), N = qmul_fma(d, c);
    const V v0 = qim(M, qdag(N));
    plq_add(sa, w, v0);
    plq_add(sd, -w, v0);
    if (RE) re += qre(M, qdag(N));
    if (B) vb = qim(b, qmul_fma(qdag(N), a));
    if (C) vc = qim(c, qmul_fma(qdag(M), d));
  }
  __device__ static V lowb(const link &a, const link &b, const link &c, const link &d) {
    return qim(b, qmul_fma(qdag(qmul_fma(d, c)), a));
  }
  __device__ static V lowc(const link &a, const link &b, const link &c, const link &d) {
    return qim(c, qmul_fma(qdag(qmul_fma(a, b)), d));
  }
  __device__ static void force(const link &, const double (&acc)[NV], double (&F)[NM]) {
#pragma unroll
    for (int k = 0; k < NM; ++k) F[k] = acc[k];
  }
};
// FP32: a term is the staple, a product of three links in FP32 (two roundings per
// component); a link's staples are summed and projected, Im(U K), in FP64, as the
// staple steps do.  Rms error of the FP32 force against 80-bit arithmetic (links of
// plaquette 0.4, 24x16x18x16): 1.68e-7, staple steps 1.70e-7; projected plaquette by
// plaquette in FP32 1.98e-7.  That form has 3 instead of 4 reals per term and 152
// instead of 164 registers: FP32 32^4 55.9 against 58.2 us a step, 48^4 271 against 278.
template <> struct PlqSU2<float> {
  using T = float;
  using link = quat<T>;
  static constexpr int NM = 3, NV = 4;
  using V = pv4<T>;
  static constexpr double DF = 2.0, RP = 8.0;
  static constexpr int lrec(int nd) { return (nd * (int)sizeof(link) / 16 | 1) * 16; }
  __device__ static V term(const link &q) { return V{{q.ar, q.ai, q.br, q.bi}}; }
  template <bool B, bool C, bool RE>
  __device__ static void plane(const link &a, const link &b, const link &c, const link &d,
                               double (&sa)[NV], double (&sd)[NV], V &vb, V &vc, double w,
                               double &) {
    static_assert(!RE, "the FP32 form takes the plaquette sum");
    const link M = qmul_fma(a, b), N = qmul_fma(d, c);
    plq_add(sa, w, term(qmul_fma(b, qdag(N))));
    plq_add(sd, w, term(qmul_fma(c, qdag(M))));
    if (B) vb = term(qmul_fma(qdag(N), a));
    if (C) vc = term(qmul_fma(qdag(M), d));
  }
  __device__ static V lowb(const link &a, const link &, const link &c, const link &d) {
    return term(qmul_fma(qdag(qmul_fma(d, c)), a));
  }
  __device__ static V lowc(const link &a, const link &b, const link &, const link &d) {
    return term(qmul_fma(qdag(qmul_fma(a, b)), d));
  }
  __device__ static void force(const link &u, const double (&K)[NV], double (&F)[NM]) {
    const pv3<double> v = qim(to_d(u), quat<double>{K[0], K[1], K[2], K[3]});
#pragma unroll
    for (int k = 0; k < NM; ++k) F[k] = v.k[k];
  }
};

// sin and cos of t = q pi/2 + r, |r| <= pi/4 (Cody and Waite, Software Manual for the
// Elementary Functions, 1980: pi/2 in two parts, the first its leading 33 bits, so that
// q times it is exact for the q < 2^17 that occur, the second the rest rounded), by
// Taylor series to the eighth power of y = r^2: cos r = c, sin r = r + r y w.  First
// terms left out, at y = (pi/4)^2: 2.1e-18 of the cosine, 1.1e-19 of the sine's.  LONG:
// the cosine's ninth power too (at y = 1 the first terms left out are 4e-19 and 8e-18).
template <bool LONG = false>
__host__ __device__ __forceinline__ void plq_series(double y, double &c, double &w) {
  double t = 1.0 / 20922789888000.0;
  if (LONG) t = fma(y, -1.0 / 6402373705728000.0, t);
  t = fma(y, t, -1.0 / 87178291200.0);
  double u = fma(y, 1.0 / 355687428096000.0, -1.0 / 1307674368000.0);
  t = fma(y, t, 1.0 / 479001600);
  u = fma(y, u, 1.0 / 6227020800.0);
  t = fma(y, t, -1.0 / 3628800);
  u = fma(y, u, -1.0 / 39916800);
  t = fma(y, t, 1.0 / 40320);
  u = fma(y, u, 1.0 / 362880);
  t = fma(y, t, -1.0 / 720);
  u = fma(y, u, -1.0 / 5040);
  t = fma(y, t, 1.0 / 24);
  u = fma(y, u, 1.0 / 120);
  t = fma(y, t, -0.5);
  u = fma(y, u, -1.0 / 6);
  c = fma(y, t, 1.0);
  w = u;
}
__host__ __device__ __forceinline__ void plq_sincos(double r, double &c, double &s) {
  const double y = r * r;
  double w;
  plq_series(y, c, w);
  s = fma(r * y, w, r);
}
__host__ __device__ __forceinline__ double plq_reduce(double a, int &j) {
  if (fabs(a) > 1e5) {
    // whole turns off first, 2 pi in two parts (the sum rounds at 2^-52, an angle of
    // this size at 2^-37; carrying the second part to the end for every angle cost U(1) 24^4 0.5 us);
    // beyond 1e15 an angle's own spacing is an eighth and more
    if (fabs(a) > 1e15) a = fmod(a, 6.283185307179586477);
    const double n = rint(a * 0.15915494309189533577);
    a = fma(-n, 2.4492935982947064e-16, fma(-n, 6.283185307179586477, a));
  }
  const double q = rint(a * 0.6366197723675813431);
  j = (int)q;
  return fma(-q, 6.07710050650619224932e-11, fma(-q, 1.57079632673412561417, a));
}
__host__ __device__ __forceinline__ void plq_quadrant(int j, double &c, double &s) {
  const double sn = (j & 1) ? c : s, cs = (j & 1) ? s : c;
  c = ((j + 1) & 2) ? -cs : cs;
  s = (j & 2) ? -sn : sn;
}

// U(1): the links of a plaquette are phases, and every link's term is the sine of
// their sum with its sign; FP32 links are added in FP64
template <typename T_> struct PlqU1 {
  using T = T_;
  using link = T;
  static constexpr int NM = 1, NV = 1;
  struct V {
    T k[1];
  };
  static constexpr double DF = 1.0, RP = 4.0;
  static constexpr int lrec(int nd) { return (nd | 1) * (int)sizeof(T); }
  template <bool RE> __device__ static T sine(T a, T b, T c, T d, double &co) {
    const double sm = (double(a) + double(b)) - double(c), th = sm - double(d);
    if constexpr (sizeof(T) == 4) {
      // a reduced argument rounded once, |r| <= pi: the FP32 functions' fast range
      const float r = (float)fma(-rint(th * 0.15915494309189533577), 6.283185307179586477, th);
      if (RE) co = cos(th);
      return sinf(r);
    } else {
      // what the last difference rounds off goes on (TwoSum): with it the angle has the two
      // roundings of a staple's, and the force's rms error against 80-bit arithmetic is
      // 2.97e-16, staple steps 3.19e-16, without it 3.58e-16 (24^4 a twentieth faster)
      const double bb = th - sm, lo = (sm - (th - bb)) - (double(d) + bb);
      int j;
      const double r = plq_reduce(th, j) + lo;
      double cs, sn;
      plq_sincos(r, cs, sn);
      plq_quadrant(j, cs, sn);
      if (RE) co = cs;
      return sn;
    }
  }
  template <bool B, bool C, bool RE>
  __device__ static void plane(link a, link b, link c, link d, double (&sa)[NV],
                               double (&sd)[NV], V &vb, V &vc, double w, double &re) {
    double co = 0.0;
    const T s = sine<RE>(a, b, c, d, co);
    if (RE) re += co;
    plq_add(sa, w, V{{s}});
    plq_add(sd, -w, V{{s}});
    if (B) vb.k[0] = s;
    if (C) vc.k[0] = -s;
  }
  __device__ static V lowb(link a, link b, link c, link d) {
    double co;
    return V{{sine<false>(a, b, c, d, co)}};
  }
  __device__ static V lowc(link a, link b, link c, link d) {
    double co;
    return V{{-sine<false>(a, b, c, d, co)}};
  }
  __device__ static void force(link, const double (&acc)[NV], double (&F)[NM]) { F[0] = acc[0]; }
};

// ------------------------------------------------------------------- memory --
__device__ __forceinline__ void plq_barrier() {
  // LDS writes done, then the barrier; global loads may stay in flight
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// fields of phases
template <typename T, typename = std::enable_if_t<std::is_floating_point<T>::value>>
__device__ __forceinline__ T *fld_add(T *p, size_t k) {
  return p + k;
}
template <typename T, typename = std::enable_if_t<std::is_floating_point<T>::value>>
__device__ __forceinline__ const T *fld_add(const T *p, size_t k) {
  return p + k;
}
template <typename T, typename = std::enable_if_t<std::is_floating_point<T>::value>>
__device__ __forceinline__ T ldq(const T *__restrict__ p, uint32_t i) {
  return ldo(p, i);
}

// The exchange in LDS: one record per thread (and of a halo row) with the nd
// links, one per thread with the 2 (nd - 1) terms.  The offsets within a record
// are immediates of the LDS instructions, so a thread needs one address per
// neighbour; records are odd multiples of 16 B (links) or 8 B apart modulo the
// banks, so the lanes of an access spread over them.
template <class G, int ND> constexpr int plq_vrec() {
  return (2 * (ND - 1) * G::NV | 1) * (int)sizeof(typename G::T);
}
__device__ __forceinline__ void plq_put(char *rec, int k, const quat<double> &q) {
  su2_d2 *p = (su2_d2 *)rec + 2 * k;
  p[0] = su2_d2{q.ar, q.ai};
  p[1] = su2_d2{q.br, q.bi};
}
__device__ __forceinline__ void plq_get(const char *rec, int k, quat<double> &q) {
  const su2_d2 *p = (const su2_d2 *)rec + 2 * k;
  const su2_d2 a = p[0], b = p[1];
  q = quat<double>{a.x, a.y, b.x, b.y};
}
__device__ __forceinline__ void plq_put(char *rec, int k, const quat<float> &q) {
  ((su2_f4 *)rec)[k] = su2_f4{q.ar, q.ai, q.br, q.bi};
}
__device__ __forceinline__ void plq_get(const char *rec, int k, quat<float> &q) {
  const su2_f4 a = ((const su2_f4 *)rec)[k];
  q = quat<float>{a.x, a.y, a.z, a.w};
}
template <typename T> __device__ __forceinline__ void plq_put(char *rec, int k, const T &q) {
  ((T *)rec)[k] = q;
}
template <typename T> __device__ __forceinline__ void plq_get(const char *rec, int k, T &q) {
  q = ((const T *)rec)[k];
}
template <class G>
__device__ __forceinline__ void plq_putv(char *rec, int k, const typename G::V &v) {
  typename G::T *p = (typename G::T *)rec + G::NV * k;
#pragma unroll
  for (int i = 0; i < G::NV; ++i) p[i] = v.k[i];
}
template <class G>
__device__ __forceinline__ void plq_getv(const char *rec, int k, typename G::V &v) {
  const typename G::T *p = (const typename G::T *)rec + G::NV * k;
#pragma unroll
  for (int i = 0; i < G::NV; ++i) v.k[i] = p[i];
}
template <class G, int ND> size_t plq_lds(const PlqGeo &g) {
  const size_t nt = plq_threads(g);
  return (nt + g.L[g.nd - 1]) * G::lrec(ND) + nt * plq_vrec<G, ND>();
}

// the values are complete here: keeps the compiler from sinking their arithmetic
// past later loads, which would hold its operands in registers
template <typename T, int N> __device__ __forceinline__ void plq_pin(T (&v)[N]) {
#pragma unroll
  for (int k = 0; k < N; ++k) asm volatile("" : "+v"(v[k]));
}

// cos a and sin(a)/a of the FP64 update for x = a^2: the series in x up to 1, beyond
// that in the square of the reduced angle
__host__ __device__ __forceinline__ void cos_sinc_fp64(double x, double &c, double &s) {
  double y = x, r = 0.0, w;
  int j = 0;
  const bool big = !(x <= 1.0);
  if (big) {
    r = plq_reduce(sqrt(x), j);
    y = r * r;
  }
  plq_series<true>(y, c, w);
  if (big) {
    s = fma(r * y, w, r);
    plq_quadrant(j, c, s);
    s = s / sqrt(x);
  } else {
    s = fma(y, w, 1.0);
  }
}

// element i + k V of a plane triple as one scalar base + 32-bit byte offset
// (3 V sizeof(T) < 2^32): the three planes share the base's registers
template <typename T> __device__ __forceinline__ uint32_t plq_off(uint32_t V, int k, uint32_t i) {
  return (i + (uint32_t)k * V) * (uint32_t)sizeof(T);
}

// momentum and link update of one link from F = Im(U K):
// P' = P - DF coef ep F rounded once, U' = exp(eu P') U
template <class G, bool W, int NT, class UO, typename T = typename G::T>
__device__ __forceinline__ void plq_update(const typename G::link &u, const double (&F)[G::NM],
                                           const T (&pi)[G::NM], T (&pn)[G::NM], T *Pw,
                                           uint32_t V, UO Uo, uint32_t s, const FusedCoef &c) {
  const double f = G::DF * c.coef * c.ep;
#pragma unroll
  for (int k = 0; k < G::NM; ++k) {
    pn[k] = T(fma(-f, F[k], double(pi[k])));
    T *q = (T *)((char *)Pw + plq_off<T>(V, k, s));
    if (NT) __builtin_nontemporal_store(pn[k], q);
    else *q = pn[k];
  }
  if constexpr (W && G::NM == 1) {
    sto_h<NT>(Uo, s, T(fma(c.eu, double(pn[0]), double(u))));
  } else if constexpr (W) {
    const double e0 = c.eu * double(pn[0]), e1 = c.eu * double(pn[1]), e2 = c.eu * double(pn[2]);
    const double x = fma(e0, e0, fma(e1, e1, e2 * e2));
    double cs, sn;
    if constexpr (sizeof(T) == 4) cos_sinc_step(x, cs, sn);
    else cos_sinc_fp64(x, cs, sn);
    quat<double> n = qmul_fma(quat<double>{cs, sn * e2, sn * e1, sn * e0}, to_d(u));
    if constexpr (sizeof(T) == 4) {
      if (c.flags & F_RESTORE) {
        // 1/sqrt(1 + d) as in md_su2_update
        const double d = fma(n.ar, n.ar, fma(n.ai, n.ai, fma(n.br, n.br, fma(n.bi, n.bi, -1.0))));
        const double r = (fabs(d) < 1e-4) ? 1.0 + d * (-0.5 + 0.375 * d) : 1.0 / sqrt(1.0 + d);
        n = qscale(r, n);
      }
    }
    stq<NT>(Uo, s, quat<T>{T(n.ar), T(n.ai), T(n.br), T(n.bi)});
  }
}

// ------------------------------------------------------------------ the step --
// W: write the new links (false: momenta alone); ACC: block partials of
// |P_in|^2, ReTr(U K) (FP64; 0 in FP32) and |P_out|^2.  pin / pout may be the same field.
// flags: F_PZERO (momenta read as zero), F_RESTORE; w_t / w_s weight the planes
// (1 where isotropic: fma with 1 is the plain sum).  GEN: the momenta are drawn
// (Philox counter of k_momenta_philox) instead of loaded.  NT: 0 ordinary
// accesses, 2 non-temporal stores and momentum loads.
// The site f of a block of nt threads; sums: this thread's part of the three.
template <class G, int ND, bool W, bool ACC, bool GEN, int NT, class UI, class UO>
__device__ __forceinline__ void plq_step(const PlqSite &f, int nt, char *smem, UI Uin, UO Uout,
                                         const typename G::T *Pin, typename G::T *Pout,
                                         const PlqGeo &g, const FusedCoef &c, double (&sums)[3]) {
  using T = typename G::T;
  using link = typename G::link;
  using Vc = typename G::V;
  constexpr int NM = G::NM, NV = G::NV;
  const int tid = (int)threadIdx.x;
  constexpr int R = ND - 2, Z = ND - 1;              // row and fastest direction
  constexpr bool X4 = ND == 4;
  const size_t V = (size_t)g.V;
  // LDS records: own, of the row above (or the halo's), of x+z; the terms' of
  // own, of the row below, of x-z
  constexpr int LREC = G::lrec(ND), VREC = plq_vrec<G, ND>();
  char *const lv0 = smem + (nt + g.L[Z]) * LREC;
  char *const lown = smem + tid * LREC, *const lrow = smem + f.lur * LREC,
             *const lz = smem + f.luz * LREC;
  char *const vown = lv0 + tid * VREC, *const vrow = lv0 + f.ldr * VREC,
             *const vz = lv0 + f.ldz * VREC;
  UI U[ND];
#pragma unroll
  for (int m = 0; m < ND; ++m) U[m] = fld_add(Uin, (size_t)m * V);
  const bool rin = f.rin, din = f.ldr >= 0;
  const bool edge = __builtin_amdgcn_readfirstlane((int)(__ballot(!din) != 0)) != 0;
  const double wt = c.w_t, ws = c.w_s;
  // the action partial is the FP64 form's (FP32 takes the plaquette sum)
  constexpr bool RE = ACC && sizeof(T) == 8;
  double re = 0.0;

  link own[ND], xl;
  Vc carry[ND];  // [1 ..]: the b terms of the planes (t, i) of the slice below
  int s = f.t0 * g.vol3 + f.o3;
  auto up_t = [&](int t) { return t == g.L[0] - 1 ? -(g.L[0] - 1) * g.vol3 : g.vol3; };
  {
    const int dt = f.t0 == 0 ? (g.L[0] - 1) * g.vol3 : -g.vol3;
    const link a = ldq(U[0], (uint32_t)(s + dt));
    const int up[4] = {0, X4 ? f.ux : f.ur, X4 ? f.ur : f.uz, f.uz};
    if (X4) xl = ldq(U[1], (uint32_t)(s + f.dx));
#pragma unroll
    for (int i = 1; i < ND; ++i) {
      own[i] = ldq(U[i], (uint32_t)s);
      const link cc = ldq(U[0], (uint32_t)(s + dt + up[i]));
      const link dd = ldq(U[i], (uint32_t)(s + dt));
      carry[i] = G::lowb(a, own[i], cc, dd);
    }
  }
  for (int t = f.t0; t < f.t1; ++t) {
    const int ut = up_t(t);
    double acc[ND][NV];
    link nx[ND], ux[ND], xlt;
    {
      // every load of the slice but the momenta's, in the order of use
      link lx[ND], lxu[ND];
      own[0] = ldq(U[0], (uint32_t)s);
      if constexpr (X4) {
        lx[0] = ldq(U[0], (uint32_t)(s + f.dx));
        xlt = ldq(U[1], (uint32_t)(s + f.dx + ut));
        lx[2] = ldq(U[2], (uint32_t)(s + f.dx));
        lxu[2] = ldq(U[1], (uint32_t)(s + f.dx + f.ur));
        lx[3] = ldq(U[3], (uint32_t)(s + f.dx));
        lxu[3] = ldq(U[1], (uint32_t)(s + f.dx + f.uz));
      }
      if (!rin) {
        // the links of the row above, where it is in another block, for the halo
        link h[ND];
#pragma unroll
        for (int m = 0; m < ND; ++m)
          if (m != R) h[m] = ldq(U[m], (uint32_t)(s + f.ur));
#pragma unroll
        for (int m = 0; m < ND; ++m)
          if (m != R) plq_put(lrow, m, h[m]);
      }
#pragma unroll
      for (int i = 1; i < ND; ++i) nx[i] = ldq(U[i], (uint32_t)(s + ut));
      if constexpr (X4) {
        ux[2] = ldq(U[2], (uint32_t)(s + f.ux));
        ux[3] = ldq(U[3], (uint32_t)(s + f.ux));
        ux[0] = ldq(U[0], (uint32_t)(s + f.ux));
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < ND; ++m) plq_put(lown, m, own[m]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 1; i < ND; ++i)
#pragma unroll
        for (int k = 0; k < NV; ++k) acc[i][k] = wt * double(carry[i].k[k]);
#pragma unroll
      for (int k = 0; k < NV; ++k) acc[0][k] = 0.0;
      if constexpr (X4) {
        plq_add(acc[0], wt, G::lowc(lx[0], xlt, own[0], xl));        // (t, x) at x-1
        plq_add(acc[2], ws, G::lowb(xl, own[2], lxu[2], lx[2]));     // (x, y)
        plq_add(acc[3], ws, G::lowb(xl, own[3], lxu[3], lx[3]));     // (x, z)
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < ND; ++m) plq_pin(acc[m]);
    }
    plq_barrier();
    T pi[ND][NM];
    link eR, e0, eRt, eZ, eRz, eX, eRx;
    {
      Vc vb, vc;
      double ret = 0.0, res = 0.0;
      link p, q;
      // (r, z): b term to U_z(x+r), c term to U_r(x+z)
      plq_get(lrow, Z, p);
      plq_get(lz, R, q);
      G::template plane<true, true, RE>(own[R], p, q, own[Z], acc[R], acc[Z],
                                         vb, vc, ws, res);
      plq_putv<G>(vown, ND - 2, vb);
      plq_putv<G>(vown, 2 * (ND - 1) - 1, vc);
      __builtin_amdgcn_sched_barrier(0);
      // (t, r): c term to U_t(x+r); (t, z): to U_t(x+z)
      plq_get(lrow, 0, q);
      G::template plane<true, true, RE>(own[0], nx[R], q, own[R], acc[0], acc[R],
                                         vb, vc, wt, ret);
      carry[R] = vb;
      plq_putv<G>(vown, 0, vc);
      __builtin_amdgcn_sched_barrier(0);
      plq_get(lz, 0, q);
      G::template plane<true, true, RE>(own[0], nx[Z], q, own[Z], acc[0], acc[Z],
                                         vb, vc, wt, ret);
      carry[Z] = vb;
      plq_putv<G>(vown, ND - 1, vc);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (X4) {
        plq_get(lrow, 1, q);
        G::template plane<false, true, RE>(own[1], ux[2], q, own[2], acc[1], acc[2],
                                           vb, vc, ws, res);
        plq_putv<G>(vown, 1, vc);
        __builtin_amdgcn_sched_barrier(0);
        plq_get(lz, 1, q);
        G::template plane<false, true, RE>(own[1], ux[3], q, own[3], acc[1], acc[3],
                                           vb, vc, ws, res);
        plq_putv<G>(vown, ND, vc);
        __builtin_amdgcn_sched_barrier(0);
        G::template plane<true, false, RE>(own[0], nx[1], ux[0], own[1], acc[0], acc[1],
                                           vb, vc, wt, ret);
        carry[1] = vb;
        __builtin_amdgcn_sched_barrier(0);
      }
      if (RE) {
        if (f.active) re += fma(wt, ret, ws * res);
        asm volatile("" : "+v"(re));
      }
#pragma unroll
      for (int m = 0; m < ND; ++m) plq_pin(acc[m]);
#pragma unroll
      for (int i = 1; i < ND; ++i) plq_pin(carry[i].k);
      // the momenta, in flight across the barrier
      if constexpr (GEN) {
#pragma unroll
        for (int m = 0; m < ND; ++m) {
          T z[4];
          philox_normals4<T>((uint32_t)(s * ND + m), (uint32_t)(c.gtraj & 0xffffffffu),
                             (uint32_t)(c.gtraj >> 32), c.gseed, z);
#pragma unroll
          for (int k = 0; k < NM; ++k) pi[m][k] = z[k];
        }
      } else if (c.flags & F_PZERO) {
#pragma unroll
        for (int m = 0; m < ND; ++m)
#pragma unroll
          for (int k = 0; k < NM; ++k) pi[m][k] = T(0);
      } else {
#pragma unroll
        for (int m = 0; m < ND; ++m) {
          const char *p = (const char *)(Pin + (size_t)(m * NM) * V);
#pragma unroll
          for (int k = 0; k < NM; ++k) {
            const T *q = (const T *)(p + plq_off<T>((uint32_t)g.V, k, (uint32_t)s));
            if constexpr (NT == 2) pi[m][k] = __builtin_nontemporal_load(q);
            else pi[m][k] = *q;
          }
        }
      }
      // links of the row below, where it is in another block (the waves that
      // hold such a row)
      if (edge) {
        const int sr = s + f.dr;
        eR = ldq(U[R], (uint32_t)sr);
        e0 = ldq(U[0], (uint32_t)sr);
        eRt = ldq(U[R], (uint32_t)(sr + ut));
        eZ = ldq(U[Z], (uint32_t)sr);
        eRz = ldq(U[R], (uint32_t)(sr + f.uz));
        if constexpr (X4) {
          eX = ldq(U[1], (uint32_t)sr);
          eRx = ldq(U[R], (uint32_t)(sr + f.ux));
        }
      }
    }
    plq_barrier();
    {
      Vc v;
      // from x-z: U_t, U_x (d = 4), U_r
      plq_getv<G>(vz, ND - 1, v);
      plq_add(acc[0], wt, v);
      if constexpr (X4) {
        plq_getv<G>(vz, ND, v);
        plq_add(acc[1], ws, v);
      }
      plq_getv<G>(vz, 2 * (ND - 1) - 1, v);
      plq_add(acc[R], ws, v);
      if (din) {
        // from x-r: U_t, U_x (d = 4), U_z
        plq_getv<G>(vrow, 0, v);
        plq_add(acc[0], wt, v);
        if constexpr (X4) {
          plq_getv<G>(vrow, 1, v);
          plq_add(acc[1], ws, v);
        }
        plq_getv<G>(vrow, ND - 2, v);
        plq_add(acc[Z], ws, v);
      }
      if (edge) {
        // the terms they give, for the lanes whose row below they are
        const double wte = din ? 0.0 : wt, wse = din ? 0.0 : ws;
        plq_add(acc[0], wte, G::lowc(e0, eRt, own[0], eR));           // (t, r): c is U_t(x)
        plq_add(acc[Z], wse, G::lowb(eR, own[Z], eRz, eZ));           // (r, z): b is U_z(x)
        if constexpr (X4)
          plq_add(acc[1], wse, G::lowc(eX, eRx, own[1], eR));         // (x, r): c is U_x(x)
      }
      __builtin_amdgcn_sched_barrier(0);
      if (f.active) {
#pragma unroll
        for (int m = 0; m < ND; ++m) {
          T pn[NM];
          double F[NM];
          G::force(own[m], acc[m], F);
          plq_update<G, W, NT>(own[m], F, pi[m], pn,
                               Pout + (size_t)(m * NM) * V, (uint32_t)g.V,
                               fld_add(Uout, (size_t)m * V), (uint32_t)s, c);
          if (ACC) {
#pragma unroll
            for (int k = 0; k < NM; ++k) {
              sums[0] = fma(double(pi[m][k]), double(pi[m][k]), sums[0]);
              sums[2] = fma(double(pn[k]), double(pn[k]), sums[2]);
            }
          }
        }
      }
      if (ACC) plq_pin(sums);
      // the next slice
#pragma unroll
      for (int i = 1; i < ND; ++i) own[i] = nx[i];
      if (X4) xl = xlt;
      s += ut;
    }
  }
  // ReTr(U K) of every link: a plaquette's 2 Re(P) once for each of its four
  if (ACC) sums[1] = G::RP * re;
}

// the three sums over the block's nt threads; thread k < 3 returns sum k
__device__ __forceinline__ double plq_block_sums(const double (&sums)[3], int nt, char *smem) {
  __syncthreads();
  double *l3 = (double *)smem;
  const int tid = (int)threadIdx.x, lane = tid & 63, wv = tid >> 6, nw = nt >> 6;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    double v = sums[k];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
    if (lane == 0) l3[k * 4 + wv] = v;
  }
  __syncthreads();
  double v = 0.0;
  if (tid < 3)
    for (int i = 0; i < nw; ++i) v += l3[tid * 4 + i];
  return v;
}

// waves per SIMD the registers are budgeted for
template <class G> constexpr int plq_occ() {
  return G::NM == 1 ? 4 : sizeof(typename G::T) == 8 ? 2 : 3;
}

template <class G, int ND, bool W, bool ACC, bool GEN, int NT, class UI, class UO>
__global__ __launch_bounds__(PLQ_NT, plq_occ<G>()) void k_md_plq(
    UI Uin, UO Uout, const typename G::T *Pin, typename G::T *Pout, PlqGeo g, FusedCoef c,
    double *__restrict__ partials, int pstride) {
  extern __shared__ __align__(16) char smem[];
  const int nt = (int)blockDim.x;
  const PlqSite f = plq_site(g, blockIdx.x, gridDim.x, threadIdx.x, (uint32_t)nt);
  double sums[3] = {0.0, 0.0, 0.0};
  plq_step<G, ND, W, ACC, GEN, NT>(f, nt, smem, Uin, Uout, Pin, Pout, g, c, sums);
  if (ACC) {
    const double v = plq_block_sums(sums, nt, smem);
    if (threadIdx.x < 3) partials[(size_t)threadIdx.x * pstride + blockIdx.x] = v;
  }
}

}  // namespace su2k
