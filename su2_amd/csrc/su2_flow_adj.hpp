// su2_flow_adj.hpp -- the pointwise part of a gradient-flow stage's adjoint, shared
// by the kernels of su2_flow.hip and su2_flow_plq.hip.
#pragma once
#include "su2_device.hpp"

namespace su2k {

using namespace su2dev;

template <typename T> struct v3 {
  T x, y, z;  // adjointsu2 (a, b, c)
};

// (a,b,c) <-> pure quaternion in storage order (Re a, Im a, Re b, Im b) = (q0, q3, q2, q1)
template <typename T> __device__ __forceinline__ quat<T> vq(const v3<T> &v) {
  return quat<T>{T(0), v.z, v.y, v.x};
}
template <typename T> __device__ __forceinline__ v3<T> im(const quat<T> &q) {
  return v3<T>{q.bi, q.br, q.ai};
}
template <typename T> __device__ __forceinline__ quat<T> qsub(const quat<T> &u, const quat<T> &v) {
  return quat<T>{u.ar - v.ar, u.ai - v.ai, u.br - v.br, u.bi - v.bi};
}
template <typename T> __device__ __forceinline__ quat<T> comm(const quat<T> &u, const quat<T> &v) {
  return qsub(qmul(u, v), qmul(v, u));
}
template <typename T> __device__ __forceinline__ quat<T> conj_by(const quat<T> &g, const quat<T> &y) {
  return qmul(qmul(g, y), qdag(g));  // g y g^+
}
template <typename T> __device__ __forceinline__ void vadd(v3<T> &a, const v3<T> &b, T s = T(1)) {
  a.x += s * b.x;
  a.y += s * b.y;
  a.z += s * b.z;
}
// ---------------------------------------------------------------------------
// pointwise part of one stage adjoint (see header) for one link: z = Z', y =
// lambda_W' in; lz (lambda_Z, accumulated) and the returned lambda_W out
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ v3<T> stage_adj_link(const v3<T> &z, const v3<T> &y, v3<T> &lz, T c) {
  const v3<T> a{c * z.x, c * z.y, c * z.z};
  const quat<T> A = vq(a), Y = vq(y);
  // J(-A) y = y - f1 [A, y] + f2 [A, [A, y]],  theta = 2|a| (|ad_A| = 2|a|)
  const T al2 = a.x * a.x + a.y * a.y + a.z * a.z;
  const T th2 = T(4) * al2;
  T f1, f2;
  if (th2 < T(1e-6)) {
    f1 = T(0.5) - th2 * T(1.0 / 24.0);
    f2 = T(1.0 / 6.0) - th2 * T(1.0 / 120.0);
  } else {
    const T th = dsqrt(th2);
    T sn, cs;
    dsincos(th, &sn, &cs);
    f1 = (T(1) - cs) / th2;
    f2 = (th - sn) / (th2 * th);
  }
  const quat<T> k1 = comm(A, Y);
  const quat<T> k2 = comm(A, k1);
  const v3<T> jy = im(quat<T>{T(0), Y.ai - f1 * k1.ai + f2 * k2.ai, Y.br - f1 * k1.br + f2 * k2.br,
                              Y.bi - f1 * k1.bi + f2 * k2.bi});
  vadd(lz, jy, c);
  // Ad(exp(A))^T y = g^+ y g
  const quat<T> g = qexp(a.x, a.y, a.z);
  return im(qmul(qmul(qdag(g), Y), g));
}


}  // namespace su2k
