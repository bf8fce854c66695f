// trilin.hpp -- geometric factors of a trilinear hexahedron formed at a node
// from the element's eight corners, for kernels that would otherwise stream
// them from memory.
//
// Corners [3][8] (x, y, z of corner a + 2b + 4c at (r, s, t) = (+-1, +-1, +-1)).
// A lane that owns the node column (r_i, s_j) keeps the corner differences
// the map's derivatives take there (init, once per element); at a plane t_k
// the derivatives, the Jacobian, the inverse by cofactors and JW = J w_i w_j
// w_k follow geometricFactorsHex3D (kernels/mesh/geometricFactorsHex3D.okl:
// 27-143), whose spectral derivatives D x of a trilinear map equal these up
// to rounding.
#pragma once
#include <hip/hip_runtime.h>

namespace nrs {

template <typename T> struct TriGeo {
  T dRB[3], dRT[3], dSB[3], dST[3], dT[3], wij;

  __device__ __forceinline__ void init(const T *__restrict__ P0, T r, T s, T wi, T wj)
  {
    const T hr0 = T(0.5) * (T(1) - r), hr1 = T(0.5) * (T(1) + r);
    const T hs0 = T(0.5) * (T(1) - s), hs1 = T(0.5) * (T(1) + s);
    wij = wi * wj;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const T *P = P0 + 8 * c;
      const T p0 = P[0], p1 = P[1], p2 = P[2], p3 = P[3], p4 = P[4], p5 = P[5], p6 = P[6], p7 = P[7];
      dRB[c] = T(0.5) * (hs0 * (p1 - p0) + hs1 * (p3 - p2));
      dRT[c] = T(0.5) * (hs0 * (p5 - p4) + hs1 * (p7 - p6));
      dSB[c] = T(0.5) * (hr0 * (p2 - p0) + hr1 * (p3 - p1));
      dST[c] = T(0.5) * (hr0 * (p6 - p4) + hr1 * (p7 - p5));
      dT[c] = T(0.5) * (hs0 * (hr0 * (p4 - p0) + hr1 * (p5 - p1)) + hs1 * (hr0 * (p6 - p2) + hr1 * (p7 - p3)));
    }
  }

  // g = rx ry rz sx sy sz tx ty tz JW at the plane t (GLL weight wk)
  __device__ __forceinline__ void at(T t, T wk, T (&g)[10]) const
  {
    const T ht0 = T(0.5) * (T(1) - t), ht1 = T(0.5) * (T(1) + t);
    const T xr = ht0 * dRB[0] + ht1 * dRT[0], yr = ht0 * dRB[1] + ht1 * dRT[1], zr = ht0 * dRB[2] + ht1 * dRT[2];
    const T xs = ht0 * dSB[0] + ht1 * dST[0], ys = ht0 * dSB[1] + ht1 * dST[1], zs = ht0 * dSB[2] + ht1 * dST[2];
    const T xt = dT[0], yt = dT[1], zt = dT[2];
    const T J = xr * (ys * zt - zs * yt) - yr * (xs * zt - zs * xt) + zr * (xs * yt - ys * xt);
    const T Jinv = T(1) / J;
    g[0] = (ys * zt - zs * yt) * Jinv;
    g[1] = -(xs * zt - zs * xt) * Jinv;
    g[2] = (xs * yt - ys * xt) * Jinv;
    g[3] = -(yr * zt - zr * yt) * Jinv;
    g[4] = (xr * zt - zr * xt) * Jinv;
    g[5] = -(xr * yt - yr * xt) * Jinv;
    g[6] = (yr * zs - zr * ys) * Jinv;
    g[7] = -(xr * zs - zr * xs) * Jinv;
    g[8] = (xr * ys - yr * xs) * Jinv;
    g[9] = J * wij * wk;
  }
};

// The operator's factors of a trilinear element without the divisions by J: at a
// node, the cofactors c_r, c_s, c_t (J grad r and so on) and 1/J give
//   [Gqr, Gqs, Gqt] = (w / J) C (C^T [qr, qs, qt]),
// 21 operations on the three derivatives of q against 33 through the six G.  In
// t, c_r = x_s x x_t and c_s = x_t x x_r are linear (x_t does not change along a
// lane's column) and c_t = x_r x x_s and J are quadratic.  LINEAR keeps their
// coefficients (24 values a lane, 14 operations a plane); otherwise the
// derivatives' (15 values, 27 operations), for FP64, where the larger set
// would spill.
template <typename T, bool LINEAR = sizeof(T) == 4> struct TriMetric {
  T m[LINEAR ? 24 : 15], wij;

  __device__ __forceinline__ void init(const T *__restrict__ P0, T r, T s, T wi, T wj)
  {
    TriGeo<T> g;
    g.init(P0, r, s, wi, wj);
    wij = g.wij;
    T mr[3], dr[3], ms[3], ds[3];   // x_r = mr + t dr, x_s = ms + t ds
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      mr[c] = T(0.5) * (g.dRT[c] + g.dRB[c]);
      dr[c] = T(0.5) * (g.dRT[c] - g.dRB[c]);
      ms[c] = T(0.5) * (g.dST[c] + g.dSB[c]);
      ds[c] = T(0.5) * (g.dST[c] - g.dSB[c]);
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const int p = (c + 1) % 3, q = (c + 2) % 3;
      if constexpr (LINEAR) {
        m[c] = ms[p] * g.dT[q] - ms[q] * g.dT[p];            // c_r = m[0..2] + t m[3..5]
        m[3 + c] = ds[p] * g.dT[q] - ds[q] * g.dT[p];
        m[6 + c] = g.dT[p] * mr[q] - g.dT[q] * mr[p];        // c_s = m[6..8] + t m[9..11]
        m[9 + c] = g.dT[p] * dr[q] - g.dT[q] * dr[p];
        m[12 + c] = mr[p] * ms[q] - mr[q] * ms[p];           // c_t = m[12..14] + t (m[15..17] + t m[18..20])
        m[15 + c] = (mr[p] * ds[q] - mr[q] * ds[p]) + (dr[p] * ms[q] - dr[q] * ms[p]);
        m[18 + c] = dr[p] * ds[q] - dr[q] * ds[p];
        m[21 + c] = g.dT[c];
      } else {
        m[c] = mr[c]; m[3 + c] = dr[c]; m[6 + c] = ms[c]; m[9 + c] = ds[c]; m[12 + c] = g.dT[c];
      }
    }
  }

  // at the plane t (GLL weight wk): cofactors c[0..2] = c_r, c[3..5] = c_s, c[6..8] = c_t, f = w / J, jw = J w
  __device__ __forceinline__ void at(T t, T wk, T (&c)[9], T &f, T &jw) const
  {
    T J;
    if constexpr (LINEAR) {
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        c[q] = m[q] + t * m[3 + q];
        c[3 + q] = m[6 + q] + t * m[9 + q];
        c[6 + q] = m[12 + q] + t * (m[15 + q] + t * m[18 + q]);
      }
      J = m[21] * c[6] + m[22] * c[7] + m[23] * c[8];
    } else {
      T xr[3], xs[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) { xr[q] = m[q] + t * m[3 + q]; xs[q] = m[6 + q] + t * m[9 + q]; }
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int a = (q + 1) % 3, b = (q + 2) % 3;
        c[q] = xs[a] * m[12 + b] - xs[b] * m[12 + a];
        c[3 + q] = m[12 + a] * xr[b] - m[12 + b] * xr[a];
        c[6 + q] = xr[a] * xs[b] - xr[b] * xs[a];
      }
      J = m[12] * c[6] + m[13] * c[7] + m[14] * c[8];
    }
    // 1 / J: the hardware's estimate (relative error 2^-23.4 in FP32, 2^-24.3 in FP64,
    // measured) and Newton steps, which square it, to an error of one rounding: equal to
    // the correctly rounded quotient for all of 4 million random J in both types.  Holds
    // where neither J nor 1 / J is subnormal: FP32 elements with sides of 1e-12 to 8e12.
    const T w = wij * wk;
    T ri;
    if constexpr (sizeof(T) == 4) {
      ri = __builtin_amdgcn_rcpf(J);
      ri = __builtin_fmaf(ri, __builtin_fmaf(-J, ri, 1.f), ri);
    } else {
      ri = __builtin_amdgcn_rcp(J);
      ri = __builtin_fma(ri, __builtin_fma(-J, ri, 1.0), ri);
      ri = __builtin_fma(ri, __builtin_fma(-J, ri, 1.0), ri);
    }
    f = w * ri;
    jw = J * w;
  }
};

}  // namespace nrs
