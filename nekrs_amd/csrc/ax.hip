// ax.hip -- element stiffness apply (Poisson / Helmholtz), its diagonal, the
// three-field block apply, and the Dirichlet mask, for gfx950.
//
// Design (one element = one (N+1)^2 slab of lanes, N=7: exactly one wave64):
//   * lane (i,j) keeps the k-pencil q(i,j,0..N) and the output pencil Aq(i,j,:)
//     in registers (the planes are unrolled), so the t-direction contractions
//     never touch LDS;
//   * the r/s contractions of plane k read the plane from LDS (one 8x8 slab
//     of doubles = 512 B), D rows/columns live in registers;
//   * ggeo streams as 6 coalesced runs of (N+1)^2 values per plane;
//   * the Dirichlet mask is fused into the store epilogue via a per-element
//     bit mask (Np bits), so the operator needs no separate mask launch.
// The other orders pack several elements per block so that whole waves are filled.
#include "common.hpp"
#include "kernels.hpp"
#include "trilin.hpp"
#include "tune.hpp"

namespace nrs {

namespace {
constexpr int kG00 = 0, kG01 = 1, kG11 = 2, kG12 = 3, kG02 = 4, kG22 = 5, kGWJ = 6;
}

#ifndef AX_WAVES_PER_EU
#define AX_WAVES_PER_EU 3
#endif

// Geometric factors are read exactly once per apply: load them non-temporally so
// they do not evict q/Aq lines that the gather-scatter reuses.
template <typename T> __device__ __forceinline__ T stream_load(const T *p)
{
  return __builtin_nontemporal_load(p);
}

// Synchronisation between the stages of one plane.  When an element is exactly
// one wave64 (NQ = 8) its LDS slabs are private to that wave, and a wave's LDS
// operations complete in issue order, so a wave-level barrier (compiler fence,
// as HIP's __syncwarp) is enough; other orders share or split waves and use
// the workgroup barrier.
template <int NQ> __device__ __forceinline__ void plane_sync()
{
  if constexpr (NQ * NQ == 64) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    __syncthreads();
  }
}

// Elements per block of a launch variant (1, 2, 4; elements in proportion at orders 1
// to 4 and 7 only): whole elements that fill the lanes of the block's waves.  An element of NQ^2 threads leaves lanes idle at
// most orders: order 5 ran 72 threads in two waves (56 %), order 9 100 in two
// (78 %); the first entry of every order fills at least 94 %.  Larger blocks than
// these would cap the registers of the high orders.  Order 7 is one element per
// wave.
template <int NQ, int MULT = 1> struct AxShape {
  static constexpr int ne()
  {
    switch (NQ) {
      case 2: return 16 * MULT;                                 // 64, 128, 256 threads
      case 3: return 7 * MULT;                                  // 63, 126, 252
      case 4: return 4 * MULT;                                  // 64, 128, 256
      case 5: return 5 * MULT;                                  // 125, 250, 500
      case 6: return MULT == 1 ? 7 : MULT == 2 ? 14 : 5;        // 252, 504, 180
      case 7: return MULT == 1 ? 5 : MULT == 2 ? 13 : 9;        // 245, 637, 441
      case 9: return MULT == 1 ? 3 : MULT == 2 ? 6 : 7;         // 243, 486, 567
      case 10: return MULT == 1 ? 5 : MULT == 2 ? 2 : 1;        // 500, 200, 100
      default: return MULT;                                     // order 7: 64, 128, 256
    }
  }
  static constexpr int NE = ne();
  static constexpr int THREADS = NQ * NQ * NE;
};

// Where the geometric factors come from: streamed one plane ahead, streamed
// all planes at once, or formed from the element corners.
enum { GEO_STREAM = 0, GEO_AHEAD = 1, GEO_CORNERS = 2 };

// -------------------------------------------------------------------------------------
// Single-field apply.  Restates ellipticPartialAxCoeffHex3D
// (kernels/elliptic/ellipticPartialAxCoeffHex3D.c:2-97) with the same arithmetic:
//   qr = sum_m D[i][m] q(m,j,k), qs = sum_m D[j][m] q(i,m,k), qt = sum_m D[k][m] q(i,j,m)
//   [Gqr,Gqs,Gqt] = lambda0 * G * [qr,qs,qt]
//   Aq = sum_m D[m][i] Gqr(m,j,k) + D[m][j] Gqs(i,m,k) + D[m][k] Gqt(i,j,m) (+ GwJ lambda1 q)
// The planes are unrolled, so the pencils are indexed at compile time (a rolled
// loop selected q(k) and the row of Aq with a compare per entry: 30 of about 190
// vector instructions a plane in FP64); the scheduling barrier keeps a plane's
// loads from being hoisted over the planes before it, which would cost the
// registers of every plane's factors.  HBM-bound at size: FP64, order 7, 32^3
// elements with the face fusion 210 us rolled, 178 us (1.074 GB, 6.0 TB/s);
// Helmholtz, order 9, 6840 elements 156 us, 92 us with the packing of AxShape.
// -------------------------------------------------------------------------------------
//
// FUSEX: the block's consecutive elements e, e+1 with fx[e] = 1 share their
// face i = N / i = 0 node for node; the interior nodes of that face are summed
// here through LDS (both copies get v_e + v_e+1, the gather-scatter's pair sum,
// bit for bit) and the caller's gather-scatter handle leaves them out.
//
// GEO_AHEAD: every plane's factors in flight before the first plane, for a mesh
// of so few elements that a wave has a SIMD to itself and waits out each
// plane's memory latency otherwise.
//
// GEO_CORNERS: trilinear elements.  The geometric factors are not read but
// formed at each node from the element's eight corners (corners [E][3][8]) and
// the GLL nodes and weights (zw [2][NQ]) by TriMetric (trilin.hpp).
template <typename T, int NQ, int MULT, bool POISSON, bool LFIELD, bool FUSEX = false, int GEO = GEO_STREAM>
__global__ void __launch_bounds__((AxShape<NQ, MULT>::THREADS),
                                  (GEO == GEO_AHEAD ? 1 : (sizeof(T) == 8 && NQ >= 9) ? 2 : AX_WAVES_PER_EU))
ax_kernel(int E, const int *__restrict__ elist, const T *__restrict__ ggeo,
          const T *__restrict__ Dg, const T *__restrict__ lam0, const T *__restrict__ lam1,
          const T *__restrict__ q, T *__restrict__ Aq, const uint32_t *__restrict__ maskBits,
          const uint8_t *__restrict__ fx = nullptr, const T *__restrict__ corners = nullptr,
          const T *__restrict__ zw = nullptr)
{
  constexpr int NE = AxShape<NQ, MULT>::NE;
  constexpr int NP = NQ * NQ * NQ, NQ2 = NQ * NQ;
  constexpr int NW = (NP + 31) / 32;
  __shared__ T s_D[NQ][NQ];
  __shared__ T s_q[NE][NQ][NQ];
  __shared__ T s_Gr[NE][NQ][NQ];
  __shared__ T s_Gs[NE][NQ][NQ];

  const int t = threadIdx.x;
  const int i = t % NQ;
  const int j = (t / NQ) % NQ;
  const int le = (NE == 1) ? 0 : t / NQ2;
  const int eidx = blockIdx.x * NE + le;
  const bool active = eidx < E;
  int64_t e = active ? (elist ? elist[eidx] : eidx) : 0;
  if (NQ2 == 64) e = __builtin_amdgcn_readfirstlane((int)e);   // wave-uniform element

  const int lid = j * NQ + i;          // lane offset inside a plane (32-bit)
  const T *qe = q + e * NP;
  const T *G = ggeo + e * 7 * NP;
  constexpr int NG = POISSON ? 6 : 7;
  constexpr int NA = (GEO == GEO_AHEAD) ? NQ : 2;   // planes of factors held
  T g[NA][7];
#define NRS_LOAD_G(k_, p_)                                                                            \
  do {                                                                                              \
    _Pragma("unroll") for (int c = 0; c < NG; ++c) g[p_][c] = stream_load(G + c * NP + (k_) * NQ2 + lid); \
  } while (0)
  T r_q[NQ], r_Aq[NQ];
#pragma unroll
  for (int k = 0; k < NQ; ++k) {
    r_q[k] = qe[k * NQ2 + lid];
    r_Aq[k] = T(0);
  }
  if constexpr (GEO == GEO_AHEAD) {
#pragma unroll
    for (int k = 0; k < NQ; ++k) NRS_LOAD_G(k, k);
  } else if constexpr (GEO == GEO_STREAM) {
    NRS_LOAD_G(0, 0);
  }

  if (t < NQ2) s_D[t / NQ][t % NQ] = Dg[t];
  __syncthreads();
  T Di[NQ], Dj[NQ], DTi[NQ], DTj[NQ];
#pragma unroll
  for (int m = 0; m < NQ; ++m) {
    Di[m] = s_D[i][m];
    Dj[m] = s_D[j][m];
    DTi[m] = s_D[m][i];
    DTj[m] = s_D[m][j];
  }

  const T l0c = LFIELD ? T(0) : lam0[0];
  const T l1c = (LFIELD || POISSON) ? T(0) : lam1[0];

  // corners: what the derivatives of the map take at this lane's (r, s), once per element
  TriMetric<T> tri;
  if constexpr (GEO == GEO_CORNERS) tri.init(corners + e * 24, zw[i], zw[j], zw[NQ + i], zw[NQ + j]);

#pragma unroll
  for (int k = 0; k < NQ; ++k) {
    const int n = k * NQ2;
    if constexpr (GEO != GEO_AHEAD) __builtin_amdgcn_sched_barrier(0);
    const int p = (GEO == GEO_AHEAD) ? k : k & 1;
    if constexpr (GEO == GEO_STREAM) {
      if (k + 1 < NQ) NRS_LOAD_G(k + 1, 1 - p);
    }
    T l0 = l0c, l1 = l1c;
    if (LFIELD) {
      l0 = lam0[e * NP + n + lid];
      if (!POISSON) l1 = lam1[e * NP + n + lid];
    }
    s_q[le][j][i] = r_q[k];
    T qt = 0;
#pragma unroll
    for (int m = 0; m < NQ; ++m) qt += Dg[k * NQ + m] * r_q[m];
    plane_sync<NQ>();

    T qr = 0, qs = 0;
#pragma unroll
    for (int m = 0; m < NQ; ++m) {
      qr += Di[m] * s_q[le][j][m];
      qs += Dj[m] * s_q[le][m][i];
    }
    T Gqr, Gqs, Gqt, gwj;
    if constexpr (GEO == GEO_CORNERS) {
      T c[9], f;
      tri.at(zw[k], zw[NQ + k], c, f, gwj);
      f *= l0;
      T v[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        v[d] = c[d] * qr; v[d] += c[3 + d] * qs; v[d] += c[6 + d] * qt;
        v[d] *= f;
      }
      Gqr = c[0] * v[0]; Gqr += c[1] * v[1]; Gqr += c[2] * v[2];
      Gqs = c[3] * v[0]; Gqs += c[4] * v[1]; Gqs += c[5] * v[2];
      Gqt = c[6] * v[0]; Gqt += c[7] * v[1]; Gqt += c[8] * v[2];
    } else {
      const T G00 = g[p][kG00], G01 = g[p][kG01], G02 = g[p][kG02];
      const T G11 = g[p][kG11], G12 = g[p][kG12], G22 = g[p][kG22];
      Gqr = G00 * qr; Gqr += G01 * qs; Gqr += G02 * qt;
      Gqs = G01 * qr; Gqs += G11 * qs; Gqs += G12 * qt;
      Gqt = G02 * qr; Gqt += G12 * qs; Gqt += G22 * qt;
      Gqr *= l0; Gqs *= l0; Gqt *= l0;
      gwj = POISSON ? T(0) : g[p][kGWJ];
    }
    s_Gr[le][j][i] = Gqr;
    s_Gs[le][j][i] = Gqs;
    plane_sync<NQ>();

    T a = 0;
#pragma unroll
    for (int m = 0; m < NQ; ++m) a += DTi[m] * s_Gr[le][j][m];
    T b = 0;
#pragma unroll
    for (int m = 0; m < NQ; ++m) b += DTj[m] * s_Gs[le][m][i];
    T ab = a + b;
    if (!POISSON) ab += gwj * l1 * r_q[k];
#pragma unroll
    for (int m = 0; m < NQ; ++m) r_Aq[m] += Dg[k * NQ + m] * Gqt;
    r_Aq[k] += ab;
    // the sums are needed only at the end: without this the compiler keeps every
    // plane's operands in registers and adds them up there
#pragma unroll
    for (int m = 0; m < NQ; ++m) asm volatile("" : "+v"(r_Aq[m]));
  }

  if constexpr (FUSEX) {
    static_assert(NE >= 2, "face fusion needs at least two elements per block");
    __shared__ T s_x[NE][2][NQ][NQ];     // [element][side: i = 0, i = N][j][k]
    const bool face = (i == 0 || i == NQ - 1) && j > 0 && j < NQ - 1;
    if (face) {
      const int side = (i == 0) ? 0 : 1;
#pragma unroll
      for (int k = 1; k < NQ - 1; ++k) s_x[le][side][j][k] = r_Aq[k];
    }
    __syncthreads();
    if (active && face) {
      if (i == NQ - 1 && le + 1 < NE && eidx + 1 < E && fx[eidx]) {
#pragma unroll
        for (int k = 1; k < NQ - 1; ++k) r_Aq[k] = r_Aq[k] + s_x[le + 1][0][j][k];
      } else if (i == 0 && le >= 1 && fx[eidx - 1]) {
#pragma unroll
        for (int k = 1; k < NQ - 1; ++k) r_Aq[k] = s_x[le - 1][1][j][k] + r_Aq[k];
      }
    }
  }
  if (!active) return;
  T *Ae = Aq + e * NP + lid;
  if (maskBits) {
    const uint32_t *mb = maskBits + e * NW;
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      const int n = k * NQ2 + lid;
      const bool masked = (mb[n >> 5] >> (n & 31)) & 1u;
      Ae[k * NQ2] = masked ? T(0) : r_Aq[k];
    }
  } else {
#pragma unroll
    for (int k = 0; k < NQ; ++k) Ae[k * NQ2] = r_Aq[k];
  }
}

// All planes' factors at once where the launch has at most one wave per SIMD
// (1024 on the chip): latency is what such a launch waits for (FP64, order 7, 64
// elements: 10.1 us one plane ahead, 6.1 us; 512 elements 12.8 and 10.7 us); with
// more waves per SIMD they hide each other's, and the registers would halve
// their number.  FP64 above order 7 would spill.
template <typename T, int NQ, int MULT> static bool ax_ahead(int E)
{
  return (sizeof(T) == 4 || NQ <= 8) && (int64_t)E * NQ * NQ <= 64 * 1024;
}

template <typename T, int NQ, int MULT>
static void launch_ax_nqm(int E, const int *elist, const T *ggeo, const T *D, const T *l0,
                          const T *l1, bool poisson, bool lfield, const T *q, T *Aq,
                          const uint32_t *maskBits, hipStream_t s)
{
  using S = AxShape<NQ, MULT>;
  const unsigned grid = (unsigned)((E + S::NE - 1) / S::NE);
  if (grid == 0) return;
  if constexpr (sizeof(T) == 4 || NQ <= 8) {
    if (ax_ahead<T, NQ, MULT>(E) && !lfield) {
      if (poisson)
        ax_kernel<T, NQ, MULT, true, false, false, GEO_AHEAD><<<grid, S::THREADS, 0, s>>>(E, elist, ggeo, D, l0, l1, q,
                                                                                          Aq, maskBits);
      else
        ax_kernel<T, NQ, MULT, false, false, false, GEO_AHEAD><<<grid, S::THREADS, 0, s>>>(E, elist, ggeo, D, l0, l1,
                                                                                           q, Aq, maskBits);
      NRS_LAUNCH_CHECK();
      return;
    }
  }
  if (poisson && !lfield)
    ax_kernel<T, NQ, MULT, true, false><<<grid, S::THREADS, 0, s>>>(E, elist, ggeo, D, l0, l1, q, Aq, maskBits);
  else if (poisson && lfield)
    ax_kernel<T, NQ, MULT, true, true><<<grid, S::THREADS, 0, s>>>(E, elist, ggeo, D, l0, l1, q, Aq, maskBits);
  else if (!poisson && !lfield)
    ax_kernel<T, NQ, MULT, false, false><<<grid, S::THREADS, 0, s>>>(E, elist, ggeo, D, l0, l1, q, Aq, maskBits);
  else
    ax_kernel<T, NQ, MULT, false, true><<<grid, S::THREADS, 0, s>>>(E, elist, ggeo, D, l0, l1, q, Aq, maskBits);
  NRS_LAUNCH_CHECK();
}

template <typename T, int NQ>
static void launch_ax_nq(int mult, int E, const int *elist, const T *ggeo, const T *D, const T *l0,
                         const T *l1, bool poisson, bool lfield, const T *q, T *Aq,
                         const uint32_t *maskBits, hipStream_t s)
{
  switch (mult) {
    case 2: launch_ax_nqm<T, NQ, 2>(E, elist, ggeo, D, l0, l1, poisson, lfield, q, Aq, maskBits, s); break;
    case 4: launch_ax_nqm<T, NQ, 4>(E, elist, ggeo, D, l0, l1, poisson, lfield, q, Aq, maskBits, s); break;
    default: launch_ax_nqm<T, NQ, 1>(E, elist, ggeo, D, l0, l1, poisson, lfield, q, Aq, maskBits, s); break;
  }
}

template <typename T>
void launch_ax_variant(int N, int mult, int E, const int *elist, const T *ggeo, const T *D,
                       const T *l0, const T *l1, bool poisson, bool lfield, const T *q, T *Aq,
                       const uint32_t *maskBits, hipStream_t s)
{
  switch (N + 1) {
#define NRS_AX_CASE(NQ_)                                                                          \
  case NQ_: launch_ax_nq<T, NQ_>(mult, E, elist, ggeo, D, l0, l1, poisson, lfield, q, Aq, maskBits, s); break;
    NRS_AX_CASE(2) NRS_AX_CASE(3) NRS_AX_CASE(4) NRS_AX_CASE(5) NRS_AX_CASE(6) NRS_AX_CASE(7)
    NRS_AX_CASE(8) NRS_AX_CASE(9) NRS_AX_CASE(10)
#undef NRS_AX_CASE
    default: throw Error(NRS_ERR_UNSUPPORTED, "Ax: order N must be 1..9");
  }
}

// Ax with the geometric factors formed from the element corners (trilinear
// elements); corners [E][24] relative to q, zw [2][N+1]
template <typename T, int NQ>
static void launch_ax_trilin_nq(int mult, int E, const T *corners, const T *zw, const T *D, const T *l0,
                                const T *l1, bool poisson, const T *q, T *Aq, const uint32_t *maskBits,
                                hipStream_t s)
{
#define NRS_AXT(M_)                                                                                   \
  {                                                                                                  \
    using S = AxShape<NQ, M_>;                                                                       \
    const unsigned grid = (unsigned)((E + S::NE - 1) / S::NE);                                       \
    if (grid == 0) return;                                                                           \
    if (poisson)                                                                                     \
      ax_kernel<T, NQ, M_, true, false, false, GEO_CORNERS><<<grid, S::THREADS, 0, s>>>(              \
          E, nullptr, nullptr, D, l0, l1, q, Aq, maskBits, nullptr, corners, zw);                    \
    else                                                                                             \
      ax_kernel<T, NQ, M_, false, false, false, GEO_CORNERS><<<grid, S::THREADS, 0, s>>>(             \
          E, nullptr, nullptr, D, l0, l1, q, Aq, maskBits, nullptr, corners, zw);                    \
  }
  switch (mult) {
    case 2: NRS_AXT(2) break;
    case 4: NRS_AXT(4) break;
    default: NRS_AXT(1) break;
  }
#undef NRS_AXT
  NRS_LAUNCH_CHECK();
}

template <typename T>
void launch_ax_trilin(int N, int E, const T *corners, const T *zw, const T *D, const T *l0, const T *l1,
                      bool poisson, const T *q, T *Aq, const uint32_t *maskBits, hipStream_t s, int mult)
{
  constexpr int type = dtype_of<T>::value;
  if (!mult) mult = tuned(TUNE_AX, N, type + kTuneCorners, E, tuned(TUNE_AX, N, type, E, 1));
  switch (N + 1) {
#define NRS_AXT_CASE(NQ_)                                                                          \
  case NQ_: launch_ax_trilin_nq<T, NQ_>(mult, E, corners, zw, D, l0, l1, poisson, q, Aq, maskBits, s); break;
    NRS_AXT_CASE(2) NRS_AXT_CASE(3) NRS_AXT_CASE(4) NRS_AXT_CASE(5) NRS_AXT_CASE(6) NRS_AXT_CASE(7)
    NRS_AXT_CASE(8) NRS_AXT_CASE(9) NRS_AXT_CASE(10)
#undef NRS_AXT_CASE
    default: throw Error(NRS_ERR_UNSUPPORTED, "Ax: order N must be 1..9");
  }
}
template void launch_ax_trilin<double>(int, int, const double *, const double *, const double *,
                                       const double *, const double *, bool, const double *, double *,
                                       const uint32_t *, hipStream_t, int);
template void launch_ax_trilin<float>(int, int, const float *, const float *, const float *, const float *,
                                      const float *, bool, const float *, float *, const uint32_t *,
                                      hipStream_t, int);

// Ax with the face fusion (N = 7, M elements per block); fx [E] relative to q
template <typename T, int M>
static void launch_ax_fused_m(int E, const T *ggeo, const T *D, const T *l0, const T *l1, bool poisson,
                              const T *q, T *Aq, const uint32_t *maskBits, const uint8_t *fx, hipStream_t s)
{
  using S = AxShape<8, M>;
  static_assert(S::NE == M, "one element per wave at N = 7");
  const unsigned grid = (unsigned)((E + S::NE - 1) / S::NE);
  if (grid == 0) return;
  if (ax_ahead<T, 8, M>(E)) {
    if (poisson)
      ax_kernel<T, 8, M, true, false, true, GEO_AHEAD><<<grid, S::THREADS, 0, s>>>(E, nullptr, ggeo, D, l0, l1, q, Aq,
                                                                                   maskBits, fx);
    else
      ax_kernel<T, 8, M, false, false, true, GEO_AHEAD><<<grid, S::THREADS, 0, s>>>(E, nullptr, ggeo, D, l0, l1, q, Aq,
                                                                                    maskBits, fx);
    NRS_LAUNCH_CHECK();
    return;
  }
  if (poisson)
    ax_kernel<T, 8, M, true, false, true><<<grid, S::THREADS, 0, s>>>(E, nullptr, ggeo, D, l0, l1, q, Aq,
                                                                      maskBits, fx);
  else
    ax_kernel<T, 8, M, false, false, true><<<grid, S::THREADS, 0, s>>>(E, nullptr, ggeo, D, l0, l1, q, Aq,
                                                                       maskBits, fx);
  NRS_LAUNCH_CHECK();
}

// nb: elements per block, the block the face-fusion flags were made for (fx[e] = 0 for e % nb = nb - 1)
template <typename T>
void launch_ax_fused(int N, int E, const T *ggeo, const T *D, const T *l0, const T *l1, bool poisson,
                     const T *q, T *Aq, const uint32_t *maskBits, const uint8_t *fx, hipStream_t s, int nb)
{
  NRS_CHECK(N == 7 && fx != nullptr, "Ax face fusion: order 7 only");
  if (nb == 2)
    launch_ax_fused_m<T, 2>(E, ggeo, D, l0, l1, poisson, q, Aq, maskBits, fx, s);
  else if (nb == 4)
    launch_ax_fused_m<T, 4>(E, ggeo, D, l0, l1, poisson, q, Aq, maskBits, fx, s);
  else
    throw Error(NRS_ERR_INVALID, "Ax face fusion: blocks of 2 or 4 elements");
}
template void launch_ax_fused<double>(int, int, const double *, const double *, const double *,
                                      const double *, bool, const double *, double *, const uint32_t *,
                                      const uint8_t *, hipStream_t, int);
template void launch_ax_fused<float>(int, int, const float *, const float *, const float *,
                                     const float *, bool, const float *, float *, const uint32_t *,
                                     const uint8_t *, hipStream_t, int);

// block shape: the autotuner's choice for (N, type), else variant 1
template <typename T>
void launch_ax(int N, int E, const int *elist, const T *ggeo, const T *D, const T *l0, const T *l1,
               bool poisson, bool lfield, const T *q, T *Aq, const uint32_t *maskBits,
               hipStream_t s)
{
  const int mult = tuned(TUNE_AX, N, dtype_of<T>::value, E, 1);
  launch_ax_variant<T>(N, mult, E, elist, ggeo, D, l0, l1, poisson, lfield, q, Aq, maskBits, s);
}
template void launch_ax_variant<double>(int, int, int, const int *, const double *, const double *,
                                        const double *, const double *, bool, bool, const double *,
                                        double *, const uint32_t *, hipStream_t);
template void launch_ax_variant<float>(int, int, int, const int *, const float *, const float *,
                                       const float *, const float *, bool, bool, const float *,
                                       float *, const uint32_t *, hipStream_t);

template void launch_ax<double>(int, int, const int *, const double *, const double *, const double *,
                                const double *, bool, bool, const double *, double *,
                                const uint32_t *, hipStream_t);
template void launch_ax<float>(int, int, const int *, const float *, const float *, const float *,
                               const float *, bool, bool, const float *, float *, const uint32_t *,
                               hipStream_t);

// -------------------------------------------------------------------------------------
// Three-field Helmholtz apply with coefficient fields.  Restates
// ellipticBlockPartialAxCoeffHex3D (kernels/elliptic/ellipticBlockPartialAxCoeffHex3D.c:2-147);
// the geometric factors are read once for the three fields.
// -------------------------------------------------------------------------------------
// Same scheme as ax_kernel: one (i,j) column per lane, the k-pencils of q and
// of the result in registers over unrolled planes, r/s contractions through LDS
// slabs, geometric factors prefetched one plane ahead and shared by the three
// fields, blocks of whole elements that fill their waves, the Dirichlet mask in
// the store (maskBits, optional).  HBM-bound in the count of bytes, held back by two
// waves per SIMD (registers): order 5, 5814 curved elements 57.8 -> 33 us (131 MB,
// 3.9 TB/s), and no mask pass.

// AxShape's blocks, smaller ones with coefficient fields at order 9 for their registers
template <int NQ, bool LFIELD> using BlockAxShape = AxShape<NQ, (NQ == 10 && LFIELD) ? 2 : 1>;
template <int NQ, bool LFIELD>
__global__ void __launch_bounds__((BlockAxShape<NQ, LFIELD>::THREADS), LFIELD ? 1 : 2)
block_ax_kernel(int E, int64_t offset, int64_t loffset, const double *__restrict__ ggeo,
                const double *__restrict__ Dg, const double *__restrict__ lam0,
                const double *__restrict__ lam1, const double *__restrict__ q,
                double *__restrict__ Aq, const uint32_t *__restrict__ maskBits)
{
  constexpr int NE = BlockAxShape<NQ, LFIELD>::NE;
  constexpr int NP = NQ * NQ * NQ, NQ2 = NQ * NQ;
  constexpr int NW = (NP + 31) / 32;
  constexpr int NF = 3;
  __shared__ double s_D[NQ][NQ];
  __shared__ double s_q[NF][NE][NQ][NQ];
  __shared__ double s_Gr[NF][NE][NQ][NQ];
  __shared__ double s_Gs[NF][NE][NQ][NQ];
  const int t = threadIdx.x;
  const int i = t % NQ, j = (t / NQ) % NQ, le = t / NQ2;
  const int eidx = blockIdx.x * NE + le;
  const bool active = eidx < E;      // inactive lanes read element 0 and store nothing
  const int64_t e = active ? eidx : 0;
  const int lid = j * NQ + i;
  double r_q[NF][NQ], r_Aq[NF][NQ];
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int k = 0; k < NQ; ++k) {
      r_q[f][k] = q[f * offset + e * NP + k * NQ2 + lid];
      r_Aq[f][k] = 0.0;
    }
  const double *G = ggeo + e * 7 * NP + lid;
  double g[2][7];
#pragma unroll
  for (int c = 0; c < 7; ++c) g[0][c] = stream_load(G + c * NP);
  if (t < NQ2) s_D[t / NQ][t % NQ] = Dg[t];
  __syncthreads();
  // D rows and columns in registers up to order 7; above, they would spill and
  // are read from LDS, once a plane for the three fields
  constexpr bool DREG = NQ <= 8;
  double Di[NQ], Dj[NQ], DTi[NQ], DTj[NQ];
  auto rows = [&]() {
#pragma unroll
    for (int m = 0; m < NQ; ++m) { Di[m] = s_D[i][m]; Dj[m] = s_D[j][m]; }
  };
  auto cols = [&]() {
#pragma unroll
    for (int m = 0; m < NQ; ++m) { DTi[m] = s_D[m][i]; DTj[m] = s_D[m][j]; }
  };
  if (DREG) { rows(); cols(); }
  const double l0c = LFIELD ? 0.0 : lam0[0];
  const double l1c = LFIELD ? 0.0 : lam1[0];

#pragma unroll
  for (int k = 0; k < NQ; ++k) {
    __builtin_amdgcn_sched_barrier(0);   // as in ax_kernel
    const int64_t id = e * NP + k * NQ2 + lid;
    const int p = k & 1;
    if (k + 1 < NQ) {
#pragma unroll
      for (int c = 0; c < 7; ++c) g[1 - p][c] = stream_load(G + c * NP + (k + 1) * NQ2);
    }
    double qt[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      s_q[f][le][j][i] = r_q[f][k];
      double a = 0.0;
#pragma unroll
      for (int m = 0; m < NQ; ++m) a += Dg[k * NQ + m] * r_q[f][m];
      qt[f] = a;
    }
    plane_sync<NQ>();
    if (!DREG) rows();
    double Gqt[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      double qr = 0.0, qs = 0.0;
#pragma unroll
      for (int m = 0; m < NQ; ++m) {
        qr += Di[m] * s_q[f][le][j][m];
        qs += Dj[m] * s_q[f][le][m][i];
      }
      const double l0 = LFIELD ? lam0[f * loffset + id] : l0c;
      s_Gr[f][le][j][i] = l0 * (g[p][kG00] * qr + g[p][kG01] * qs + g[p][kG02] * qt[f]);
      s_Gs[f][le][j][i] = l0 * (g[p][kG01] * qr + g[p][kG11] * qs + g[p][kG12] * qt[f]);
      Gqt[f] = l0 * (g[p][kG02] * qr + g[p][kG12] * qs + g[p][kG22] * qt[f]);
    }
    plane_sync<NQ>();
    if (!DREG) cols();
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const double l1 = LFIELD ? lam1[f * loffset + id] : l1c;
      double a = 0.0, b = 0.0;
#pragma unroll
      for (int m = 0; m < NQ; ++m) {
        a += DTi[m] * s_Gr[f][le][j][m];
        b += DTj[m] * s_Gs[f][le][m][i];
      }
      const double ab = a + b + g[p][kGWJ] * l1 * r_q[f][k];
#pragma unroll
      for (int m = 0; m < NQ; ++m) r_Aq[f][m] += Dg[k * NQ + m] * Gqt[f];
      r_Aq[f][k] += ab;
    }
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int m = 0; m < NQ; ++m) asm volatile("" : "+v"(r_Aq[f][m]));   // as in ax_kernel
  }
  if (!active) return;
  const uint32_t *mb = maskBits ? maskBits + e * NW : nullptr;
#pragma unroll
  for (int k = 0; k < NQ; ++k) {
    const int n = k * NQ2 + lid;
    const bool masked = mb && ((mb[n >> 5] >> (n & 31)) & 1u);
#pragma unroll
    for (int f = 0; f < NF; ++f) Aq[f * offset + e * NP + n] = masked ? 0.0 : r_Aq[f][k];
  }
}

void launch_block_ax(int N, int E, int64_t offset, int64_t loffset, const double *ggeo,
                     const double *D, const double *l0, const double *l1, const double *q,
                     double *Aq, hipStream_t s, bool lfield, const uint32_t *maskBits)
{
#define BLK1(NQ, LF)                                                                         \
  {                                                                                          \
    using S = BlockAxShape<NQ, LF>;                                                          \
    const unsigned g = (unsigned)((E + S::NE - 1) / S::NE);                                  \
    if (g)                                                                                   \
      block_ax_kernel<NQ, LF><<<g, S::THREADS, 0, s>>>(E, offset, loffset, ggeo, D, l0, l1, q, Aq, maskBits); \
  }
#define BLK(NQ)                                                                              \
  case NQ:                                                                                   \
    if (lfield) BLK1(NQ, true) else BLK1(NQ, false)                                          \
    break;
  switch (N + 1) {
    BLK(2) BLK(3) BLK(4) BLK(5) BLK(6) BLK(7) BLK(8) BLK(9) BLK(10)
    default: throw Error(NRS_ERR_UNSUPPORTED, "block Ax: order N must be 1..9");
  }
#undef BLK
#undef BLK1
  NRS_LAUNCH_CHECK();
}

// -------------------------------------------------------------------------------------
// Element diagonal.  Restates ellipticBlockBuildDiagonalHex3D
// (kernels/elliptic/ellipticBlockBuildDiagonalHex3D.okl:27-117) for one field:
//   diag = 2 l0 (G01 D_ii D_jj + G02 D_ii D_kk + G12 D_jj D_kk)
//        + sum_m [G00 l0](m,j,k) D_mi^2 + [G11 l0](i,m,k) D_mj^2 + [G22 l0](i,j,m) D_mk^2
//        (+ GwJ l1).  Setup-time kernel: one thread per node.
// -------------------------------------------------------------------------------------
template <typename T>
__global__ void build_diag_kernel(int N, int E, const T *__restrict__ ggeo, const T *__restrict__ D,
                                  const T *__restrict__ lam0, const T *__restrict__ lam1,
                                  int poisson, int lfield, T *__restrict__ diag)
{
  const int Nq = N + 1, Np = Nq * Nq * Nq;
  const int64_t gid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (gid >= (int64_t)E * Np) return;
  const int64_t e = gid / Np;
  const int n = (int)(gid - e * Np);
  const int i = n % Nq, j = (n / Nq) % Nq, k = n / (Nq * Nq);
  const T *G = ggeo + e * 7 * Np;
  auto L0 = [&](int nn) { return lfield ? lam0[e * Np + nn] : lam0[0]; };
  const T l0 = L0(n);
  T r = 0;
  r += T(2) * G[kG01 * Np + n] * l0 * D[i * Nq + i] * D[j * Nq + j];
  r += T(2) * G[kG02 * Np + n] * l0 * D[i * Nq + i] * D[k * Nq + k];
  r += T(2) * G[kG12 * Np + n] * l0 * D[j * Nq + j] * D[k * Nq + k];
  for (int m = 0; m < Nq; ++m) {
    const int nr = m + Nq * (j + Nq * k), ns = i + Nq * (m + Nq * k), nt = i + Nq * (j + Nq * m);
    r += G[kG00 * Np + nr] * L0(nr) * D[m * Nq + i] * D[m * Nq + i];
    r += G[kG11 * Np + ns] * L0(ns) * D[m * Nq + j] * D[m * Nq + j];
    r += G[kG22 * Np + nt] * L0(nt) * D[m * Nq + k] * D[m * Nq + k];
  }
  if (!poisson) r += G[kGWJ * Np + n] * (lfield ? lam1[gid] : lam1[0]);
  diag[gid] = r;
}

template <typename T>
void launch_build_diag(int N, int E, const T *ggeo, const T *D, const T *l0, const T *l1,
                       bool poisson, bool lfield, T *diag, hipStream_t s)
{
  const int64_t n = (int64_t)E * (N + 1) * (N + 1) * (N + 1);
  if (n == 0) return;
  build_diag_kernel<T><<<grid_for(n, 256, 1ll << 30), 256, 0, s>>>(N, E, ggeo, D, l0, l1, poisson,
                                                                   lfield, diag);
  NRS_LAUNCH_CHECK();
}
template void launch_build_diag<double>(int, int, const double *, const double *, const double *,
                                        const double *, bool, bool, double *, hipStream_t);
template void launch_build_diag<float>(int, int, const float *, const float *, const float *,
                                       const float *, bool, bool, float *, hipStream_t);

// -------------------------------------------------------------------------------------
// mask (kernels/core/mask.okl:27-35)
// -------------------------------------------------------------------------------------
template <typename T>
__global__ void mask_kernel(int64_t Nm, const int *__restrict__ ids, T *__restrict__ v)
{
  for (int64_t n = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; n < Nm;
       n += (int64_t)gridDim.x * blockDim.x)
    v[ids[n]] = T(0);
}

template <typename T>
void launch_mask(int64_t Nm, const int *ids, T *v, hipStream_t s)
{
  if (Nm <= 0) return;
  mask_kernel<T><<<grid_for(Nm, 256, 8192), 256, 0, s>>>(Nm, ids, v);
  NRS_LAUNCH_CHECK();
}
template void launch_mask<double>(int64_t, const int *, double *, hipStream_t);
template void launch_mask<float>(int64_t, const int *, float *, hipStream_t);

}  // namespace nrs
