// su2_flow_plq.hip -- one stage of the gradient-flow adjoint (the header of
// su2_flow.hip) in one pass, SU(2), d = 4, FP32: the Hessian-vector product of
// stage st completes lambda_W, and the pointwise adjoint of the stage before it
// runs on that in registers.
//
// A plaquette's four role gradients go to its four links, as the force terms of
// su2_md_plq.hpp do, so the layout is that one's: registers along t, LDS along the
// two fastest directions, the terms from x-1 evaluated again.  The two-pass form
// (k_flow_vjp_plaq, k_flow_gather_stage_adj) sends the b and c roles through a
// scratch of 36 reals per site: 245 MB of fields per stage at 24^4 instead of 101.
// The vector parts are written out: with P = (p0, p) and the pure Omega = (0, w),
//   Im(P Om) = p0 w + p x w,  Im(Om P) = p0 w - p x w,  Im([T, P]) = 2 T x p,
// and g y g^+ = (g0^2 - |g|^2) y + 2 (g.y) g + 2 g0 g x y (no |g| = 1 assumed).
//
// lambda_Z is kept as records of four reals per link (one load), in two buffers in
// turn: neighbours of a link read its old value.
//
// Bound by instruction issue (about 2000 per site and slice) with three waves per
// SIMD to cover the latencies: 157 registers, where an edge row's links are loaded in
// two trips inside their branch (carried across the barrier they cost 70 spills).
// One stage, two-pass form -> this: 24^4 57.2 -> 38.1 us (2.6 TB/s of the 101 MB),
// 32^4 181.6 -> 109.7, 20x18x15x27 31.2 -> 22.3, 16^4 21.7 -> 14.0, 12^4 19.7 -> 12.0, 8^4 18.1 ->
// 10.3; planes y z of few sites, which leave most lanes idle, keep the two passes where
// there are many (a stage with its share of the forward pass, this / two passes: 64 5 5 64
// 58 / 54, 64 2 2 64 38 / 35, 128 1 2 256 113 / 47 us; 64 6 6 64 65 / 67, 32 5 5 32 39 / 45, 32 2 2 32 23 /
// 27 us).  FP64 keeps the two passes: its registers would not fit two waves.
#include "su2_flow_adj.hpp"
#include "su2_md_plq.hpp"

namespace su2k {

namespace {

constexpr int CUS = 256;
constexpr int FLP_LREC = 112;  // 4 links of 16 B, 4 cotangents of 12 B: 7 (odd) times 16 B
constexpr int FLP_VREC = 76;   // 6 terms of 12 B, an odd number of dwords

size_t flp_lds(const PlqGeo &g) {
  const size_t nt = plq_threads(g);
  return (nt + g.L[3]) * FLP_LREC + nt * FLP_VREC;
}

// vectors in the order (Im a, Re b, Im b) of the quaternion's imaginary part
struct w3 {
  float x, y, z;
};
__device__ __forceinline__ w3 operator+(w3 a, w3 b) { return w3{a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ w3 operator-(w3 a, w3 b) { return w3{a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ w3 scl(float f, w3 a) { return w3{f * a.x, f * a.y, f * a.z}; }
__device__ __forceinline__ w3 madd(float f, w3 a, w3 b) {
  return w3{fmaf(f, a.x, b.x), fmaf(f, a.y, b.y), fmaf(f, a.z, b.z)};
}
// c + a x b
__device__ __forceinline__ w3 cross_add(w3 a, w3 b, w3 c) {
  return w3{fmaf(a.y, b.z, fmaf(-a.z, b.y, c.x)), fmaf(a.z, b.x, fmaf(-a.x, b.z, c.y)),
            fmaf(a.x, b.y, fmaf(-a.y, b.x, c.z))};
}
__device__ __forceinline__ w3 vec(const quat<float> &q) { return w3{q.ai, q.br, q.bi}; }
// g y g^+ (sg = 1) or g^+ y g (sg = -1)
__device__ __forceinline__ w3 turn(const quat<float> &g, w3 y, float sg) {
  const w3 q = vec(g);
  const float qq = fmaf(q.x, q.x, fmaf(q.y, q.y, q.z * q.z));
  const float qy = fmaf(q.x, y.x, fmaf(q.y, y.y, q.z * y.z));
  const float g0 = 2.0f * sg * g.ar;
  return cross_add(scl(g0, q), y, madd(2.0f * qy, q, scl(fmaf(g.ar, g.ar, -qq), y)));
}

// a link with its cotangent
struct lc {
  quat<float> u;
  w3 l;
};

// the role gradients of a plaquette's links a, b, c, d (bits of WANT: 1 a and d,
// 2 b, 4 c)
struct Roles {
  w3 a, b, c, d;
};
template <int WANT>
__device__ __forceinline__ void hvp_plane(const lc &a, const lc &b, const lc &c, const lc &d,
                                          Roles &r) {
  const quat<float> P = qmul_fma(qmul_fma(a.u, b.u), qdag(qmul_fma(d.u, c.u)));
  const w3 p = vec(P);
  const w3 tb = turn(a.u, b.l, 1.0f), mtc = turn(d.u, c.l, 1.0f);  // T_b, -T_c
  const w3 w = ((a.l + tb) - mtc) - d.l;
  if (WANT & 1) {
    r.a = cross_add(p, madd(-2.0f, tb, w), scl(P.ar, w));
    r.d = cross_add(p, madd(2.0f, mtc, w), scl(-P.ar, w));
  }
  if (WANT & 2) r.b = turn(a.u, cross_add(p, w, scl(P.ar, w)), -1.0f);
  if (WANT & 4) r.c = turn(d.u, cross_add(p, w, scl(-P.ar, w)), -1.0f);
}

__device__ __forceinline__ void flp_put(char *rec, int k, const lc &q) {
  plq_put(rec, k, q.u);
  float *p = (float *)(rec + 64) + 3 * k;
  p[0] = q.l.x;
  p[1] = q.l.y;
  p[2] = q.l.z;
}
__device__ __forceinline__ void flp_get(const char *rec, int k, lc &q) {
  plq_get(rec, k, q.u);
  const float *p = (const float *)(rec + 64) + 3 * k;
  q.l = w3{p[0], p[1], p[2]};
}
__device__ __forceinline__ void flp_putv(char *rec, int k, w3 v) {
  float *p = (float *)rec + 3 * k;
  p[0] = v.x;
  p[1] = v.y;
  p[2] = v.z;
}
__device__ __forceinline__ w3 flp_getv(const char *rec, int k) {
  const float *p = (const float *)rec + 3 * k;
  return w3{p[0], p[1], p[2]};
}
__device__ __forceinline__ void flp_add(float (&acc)[3], float w, w3 v) {
  acc[0] = fmaf(w, v.x, acc[0]);
  acc[1] = fmaf(w, v.y, acc[1]);
  acc[2] = fmaf(w, v.z, acc[2]);
}

// stage_adj_link in vector form.  With x = |A|, y = x^2, C = cos x, S = sin x / x:
// exp(A) = (C, S A), f1 = (1 - cos 2x) / (2x)^2 = S^2 / 2 and
// f2 = (2x - sin 2x) / (2x)^3 = sum_k (-4y)^k / (2k+3)!, so three Taylor series in
// y (truncated below 1e-8 for y <= 1) stand for two sine/cosine calls, two roots and
// four divisions; |A| > 1 takes stage_adj_link itself.
__device__ __forceinline__ w3 flp_adj_link(w3 z, w3 yw, w3 &lz, float c) {
  const w3 a = scl(c, z);
  const float y = fmaf(a.x, a.x, fmaf(a.y, a.y, a.z * a.z));
  if (!(y <= 1.0f)) {
    v3<float> l{lz.z, lz.y, lz.x};
    const v3<float> r = stage_adj_link<float>(v3<float>{z.z, z.y, z.x}, v3<float>{yw.z, yw.y, yw.x}, l, c);
    lz = w3{l.z, l.y, l.x};
    return w3{r.z, r.y, r.x};
  }
  constexpr float C6 = 1.0f / 479001600.0f, C5 = -1.0f / 3628800.0f, C4 = 1.0f / 40320.0f,
                  C3 = -1.0f / 720.0f, C2 = 1.0f / 24.0f;
  constexpr float S5 = -1.0f / 39916800.0f, S4 = 1.0f / 362880.0f, S3 = -1.0f / 5040.0f,
                  S2 = 1.0f / 120.0f, S1 = -1.0f / 6.0f;
  constexpr float G6 = 4096.0f / 1307674368000.0f, G5 = -1024.0f / 6227020800.0f,
                  G4 = 256.0f / 39916800.0f, G3 = -64.0f / 362880.0f, G2 = 16.0f / 5040.0f,
                  G1 = -4.0f / 120.0f, G0 = 1.0f / 6.0f;
  const float cs = fmaf(y, fmaf(y, fmaf(y, fmaf(y, fmaf(y, fmaf(y, C6, C5), C4), C3), C2), -0.5f), 1.0f);
  const float sn = fmaf(y, fmaf(y, fmaf(y, fmaf(y, fmaf(y, S5, S4), S3), S2), S1), 1.0f);
  const float f2 =
      fmaf(y, fmaf(y, fmaf(y, fmaf(y, fmaf(y, fmaf(y, G6, G5), G4), G3), G2), G1), G0);
  const w3 zero{0.f, 0.f, 0.f};
  const w3 k = cross_add(a, yw, zero), kk = cross_add(a, k, zero);  // [A,Y]/2, [A,[A,Y]]/4
  lz = madd(c, madd(4.0f * f2, kk, madd(-sn * sn, k, yw)), lz);
  return turn(quat<float>{cs, sn * a.x, sn * a.y, sn * a.z}, yw, -1.0f);
}

// lamW += b (dD/dW)^T lambda_Z; with NEXT then the pointwise adjoint of the stage
// with Z' = Zs and coefficient c: lambda_Z (0 with zero_lamZ) to lzo, lambda_W in place
template <bool NEXT>
__global__ __launch_bounds__(PLQ_NT, 3) void k_flow_hvp_plq(
    const quat<float> *__restrict__ Uin, const su2_f4 *__restrict__ lzi, su2_f4 *__restrict__ lzo,
    float *__restrict__ lamW, const float *__restrict__ Zs, PlqGeo g, float fb, float wt,
    float ws, float cz, int zero_lamZ) {
  extern __shared__ __align__(16) char smem[];
  constexpr int R = 2, Z = 3;
  const int nt = (int)blockDim.x, tid = (int)threadIdx.x;
  const PlqSite f = plq_site(g, blockIdx.x, gridDim.x, (uint32_t)tid, (uint32_t)nt);
  const uint32_t V = (uint32_t)g.V;
  char *const lv0 = smem + (nt + g.L[Z]) * FLP_LREC;
  char *const lown = smem + tid * FLP_LREC, *const lrow = smem + f.lur * FLP_LREC,
             *const lz0 = smem + f.luz * FLP_LREC;
  char *const vown = lv0 + tid * FLP_VREC, *const vrow = lv0 + f.ldr * FLP_VREC,
             *const vz = lv0 + f.ldz * FLP_VREC;
  const bool rin = f.rin, din = f.ldr >= 0;
  const bool edge = __builtin_amdgcn_readfirstlane((int)(__ballot(!din) != 0)) != 0;
  auto ld = [&](int m, int i) {
    lc q;
    q.u = ldo(Uin + (size_t)m * V, (uint32_t)i);
    const su2_f4 l = ldo(lzi + (size_t)m * V, (uint32_t)i);
    q.l = w3{l.x, l.y, l.z};
    return q;
  };
  lc own[4], xl;
  w3 carry[4];
  int s = f.t0 * g.vol3 + f.o3;
  Roles r;
  {
    const int dt = f.t0 == 0 ? (g.L[0] - 1) * g.vol3 : -g.vol3;
    const lc a = ld(0, s + dt);
    const int up[4] = {0, f.ux, f.ur, f.uz};
    xl = ld(1, s + f.dx);
#pragma unroll
    for (int i = 1; i < 4; ++i) {
      own[i] = ld(i, s);
      hvp_plane<2>(a, own[i], ld(0, s + dt + up[i]), ld(i, s + dt), r);
      carry[i] = r.b;
    }
  }
  for (int t = f.t0; t < f.t1; ++t) {
    const int ut = t == g.L[0] - 1 ? -(g.L[0] - 1) * g.vol3 : g.vol3;
    float acc[4][3];
    lc nx[4], ux[4], xlt;
    {
      lc lx[4], lxu[4];
      own[0] = ld(0, s);
      lx[0] = ld(0, s + f.dx);
      xlt = ld(1, s + f.dx + ut);
      lx[2] = ld(2, s + f.dx);
      lxu[2] = ld(1, s + f.dx + f.ur);
      lx[3] = ld(3, s + f.dx);
      lxu[3] = ld(1, s + f.dx + f.uz);
      if (!rin) {
        const lc h0 = ld(0, s + f.ur), h1 = ld(1, s + f.ur), h3 = ld(3, s + f.ur);
        flp_put(lrow, 0, h0);
        flp_put(lrow, 1, h1);
        flp_put(lrow, 3, h3);
      }
#pragma unroll
      for (int i = 1; i < 4; ++i) nx[i] = ld(i, s + ut);
      ux[2] = ld(2, s + f.ux);
      ux[3] = ld(3, s + f.ux);
      ux[0] = ld(0, s + f.ux);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < 4; ++m) flp_put(lown, m, own[m]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < 4; ++m) acc[m][0] = acc[m][1] = acc[m][2] = 0.0f;
#pragma unroll
      for (int i = 1; i < 4; ++i) flp_add(acc[i], wt, carry[i]);
      hvp_plane<4>(lx[0], xlt, own[0], xl, r);
      flp_add(acc[0], wt, r.c);
      hvp_plane<2>(xl, own[2], lxu[2], lx[2], r);
      flp_add(acc[2], ws, r.b);
      hvp_plane<2>(xl, own[3], lxu[3], lx[3], r);
      flp_add(acc[3], ws, r.b);
#pragma unroll
      for (int m = 0; m < 4; ++m) plq_pin(acc[m]);
    }
    plq_barrier();
    w3 y[4], z[4];
    {
      lc p, q;
      auto both = [&](int i, int j, float w) {
        flp_add(acc[i], w, r.a);
        flp_add(acc[j], w, r.d);
      };
      flp_get(lrow, Z, p);
      flp_get(lz0, R, q);
      hvp_plane<7>(own[R], p, q, own[Z], r);
      both(R, Z, ws);
      flp_putv(vown, 2, r.b);
      flp_putv(vown, 5, r.c);
      __builtin_amdgcn_sched_barrier(0);
      flp_get(lrow, 0, q);
      hvp_plane<7>(own[0], nx[R], q, own[R], r);
      both(0, R, wt);
      carry[R] = r.b;
      flp_putv(vown, 0, r.c);
      __builtin_amdgcn_sched_barrier(0);
      flp_get(lz0, 0, q);
      hvp_plane<7>(own[0], nx[Z], q, own[Z], r);
      both(0, Z, wt);
      carry[Z] = r.b;
      flp_putv(vown, 3, r.c);
      __builtin_amdgcn_sched_barrier(0);
      flp_get(lrow, 1, q);
      hvp_plane<5>(own[1], ux[R], q, own[R], r);
      both(1, R, ws);
      flp_putv(vown, 1, r.c);
      __builtin_amdgcn_sched_barrier(0);
      flp_get(lz0, 1, q);
      hvp_plane<5>(own[1], ux[Z], q, own[Z], r);
      both(1, Z, ws);
      flp_putv(vown, 4, r.c);
      __builtin_amdgcn_sched_barrier(0);
      hvp_plane<3>(own[0], nx[1], ux[0], own[1], r);
      both(0, 1, wt);
      carry[1] = r.b;
#pragma unroll
      for (int m = 0; m < 4; ++m) plq_pin(acc[m]);
#pragma unroll
      for (int i = 1; i < 4; ++i)
        asm volatile("" : "+v"(carry[i].x), "+v"(carry[i].y), "+v"(carry[i].z));
      __builtin_amdgcn_sched_barrier(0);
    }
    plq_barrier();
    {
      flp_add(acc[0], wt, flp_getv(vz, 3));
      flp_add(acc[1], ws, flp_getv(vz, 4));
      flp_add(acc[R], ws, flp_getv(vz, 5));
      if (din) {
        flp_add(acc[0], wt, flp_getv(vrow, 0));
        flp_add(acc[1], ws, flp_getv(vrow, 1));
        flp_add(acc[Z], ws, flp_getv(vrow, 2));
      }
      if (edge) {
        const float wte = din ? 0.0f : wt, wse = din ? 0.0f : ws;
        const int sr = s + f.dr;
        const lc eR = ld(R, sr);
        {
          const lc e0 = ld(0, sr), eRt = ld(R, sr + ut);
          hvp_plane<4>(e0, eRt, own[0], eR, r);
          flp_add(acc[0], wte, r.c);
          plq_pin(acc[0]);
          __builtin_amdgcn_sched_barrier(0);
        }
        const lc eZ = ld(Z, sr), eRz = ld(R, sr + f.uz), eX = ld(1, sr), eRx = ld(R, sr + f.ux);
        hvp_plane<2>(eR, own[Z], eRz, eZ, r);
        flp_add(acc[Z], wse, r.b);
        hvp_plane<4>(eX, eRx, own[1], eR, r);
        flp_add(acc[1], wse, r.c);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const char *pw = (const char *)(lamW + (size_t)(m * 3) * V);
        y[m] = w3{*(const float *)(pw + plq_off<float>(V, 2, s)),
                  *(const float *)(pw + plq_off<float>(V, 1, s)),
                  *(const float *)(pw + plq_off<float>(V, 0, s))};
        if (NEXT) {
          const char *pz = (const char *)(Zs + (size_t)(m * 3) * V);
          z[m] = w3{*(const float *)(pz + plq_off<float>(V, 2, s)),
                    *(const float *)(pz + plq_off<float>(V, 1, s)),
                    *(const float *)(pz + plq_off<float>(V, 0, s))};
        }
      }
      if (f.active) {
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          // planes hold (a, b, c) = (Im b, Re b, Im a)
          w3 yw{fmaf(fb, acc[m][0], y[m].x), fmaf(fb, acc[m][1], y[m].y),
                fmaf(fb, acc[m][2], y[m].z)};
          if (NEXT) {
            w3 lz = zero_lamZ ? w3{0.f, 0.f, 0.f} : own[m].l;
            yw = flp_adj_link(z[m], yw, lz, cz);
            sto(lzo + (size_t)m * V, (uint32_t)s, su2_f4{lz.x, lz.y, lz.z, 0.f});
          }
          char *pw = (char *)(lamW + (size_t)(m * 3) * V);
          *(float *)(pw + plq_off<float>(V, 0, s)) = yw.z;
          *(float *)(pw + plq_off<float>(V, 1, s)) = yw.y;
          *(float *)(pw + plq_off<float>(V, 2, s)) = yw.x;
        }
      }
#pragma unroll
      for (int i = 1; i < 4; ++i) own[i] = nx[i];
      xl = xlt;
      s += ut;
    }
  }
}

// the first stage adjoint of a backward pass: pointwise, lambda_Z from zero into
// the record layout
__global__ __launch_bounds__(PLQ_NT) void k_flow_first_adj(const float *__restrict__ Zs,
                                                         float *__restrict__ lamW,
                                                         su2_f4 *__restrict__ lzo, int V, float c) {
  const int i = blockIdx.x * PLQ_NT + threadIdx.x;
  if (i >= 4 * V) return;
  const int mu = i / V, s = i - mu * V;
  float *w = lamW + (size_t)(mu * 3) * V + s;
  const float *z = Zs + (size_t)(mu * 3) * V + s;
  w3 lz{0.f, 0.f, 0.f};
  const w3 y = flp_adj_link(w3{z[2 * (size_t)V], z[V], z[0]}, w3{w[2 * (size_t)V], w[V], w[0]}, lz, c);
  lzo[i] = su2_f4{lz.x, lz.y, lz.z, 0.f};
  w[0] = y.z;
  w[V] = y.y;
  w[2 * (size_t)V] = y.x;
}

bool flp_geo(const Geo &geo, PlqGeo &g) {
  if (geo.nd != 4 || !make_plq_rows(geo.L, 4, geo.V, g) || !plq_full(g)) return false;
  const int waves = (int)plq_threads(g) / 64;
  return make_plq_chunks(std::max(1, std::min(12 / waves, (int)(160 * 1024 / flp_lds(g)))), CUS, g);
}

}  // namespace

bool flow_fused_ok(int prec, const Geo &geo) {
  PlqGeo g;
  return prec == 1 && flp_geo(geo, g);
}

void launch_flow_first_adj(const void *Zs, void *lamW, void *lzo, const Geo &geo, double c,
                           hipStream_t st) {
  hipLaunchKernelGGL(k_flow_first_adj, dim3((unsigned)((4 * (long)geo.V + PLQ_NT - 1) / PLQ_NT)),
                     dim3(PLQ_NT), 0, st, (const float *)Zs, (float *)lamW, (su2_f4 *)lzo, geo.V,
                     (float)c);
}

void launch_flow_fused(const void *U, const void *lzi, void *lzo, void *lamW, const void *Zs,
                       const Geo &geo, double b, double w_t, double w_s, double c, int zero_lamZ,
                       hipStream_t st) {
  PlqGeo g;
  if (!flp_geo(geo, g)) return;
  const dim3 grid(plq_blocks(g)), block(plq_threads(g));
  const unsigned lds = (unsigned)flp_lds(g);
  if (Zs)
    hipLaunchKernelGGL((k_flow_hvp_plq<true>), grid, block, lds, st, (const quat<float> *)U,
                       (const su2_f4 *)lzi, (su2_f4 *)lzo, (float *)lamW, (const float *)Zs, g,
                       (float)(2.0 * b), (float)w_t, (float)w_s, (float)c, zero_lamZ);
  else
    hipLaunchKernelGGL((k_flow_hvp_plq<false>), grid, block, lds, st, (const quat<float> *)U,
                       (const su2_f4 *)lzi, (su2_f4 *)lzo, (float *)lamW, (const float *)Zs, g,
                       (float)(2.0 * b), (float)w_t, (float)w_s, (float)c, zero_lamZ);
}

}  // namespace su2k
