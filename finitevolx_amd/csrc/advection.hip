// Fused flux-form advection tendency (Advection2D.__call__,
// advection/advection.py:329-420) for every reconstruction the drop-in
// exposes: naive, upwind1/2/3, weno3, wenoz3, weno5, wenoz5 and the four TVD
// limiters, unmasked or with per-face stencil tiers (advection/flux.py:100-253).
//
// One pass per wavefront tile (advection_kernel): the tracer column of each
// lane plus a 3-cell halo sits in registers, loaded from coalesced rows;
// every face flux of the tile is reconstructed exactly once (one
// upwind-selected, branch-free evaluation per face, the reference evaluates
// both branches); the flux divergence, the mask and the zero 2-cell output
// ring are applied in the same kernel.  HBM traffic per cell: read h, u, v
// and write the tendency (+ 2 tier bytes + 1 mask byte masked).

#include <algorithm>
#include <cmath>
#include <mutex>

#include "fvx_common.hpp"

namespace fvx {

enum AdvMethod : int {
  kNaive = 0,
  kUpwind1 = 1,
  kUpwind2 = 2,
  kUpwind3 = 3,
  kWeno3 = 4,
  kWenoZ3 = 5,
  kWeno5 = 6,
  kWenoZ5 = 7,
  kTvd = 8,
};
enum Limiter : int { kMinmod = 0, kVanLeer = 1, kSuperbee = 2, kMC = 3 };

// --- point reconstructions (advection/weno.py) -----------------------------
//
// The nonlinear weights are the reference's; only how they are divided out
// differs, because the divisions dominate the instruction count of these
// VALU-bound kernels.  FP32: each division is a product with the hardware
// reciprocal (v_rcp_f32, 1 ulp), inside the FP32 stencils' 1e-5 bound.  FP64:
// the normalised combination sum_k w_k q_k / sum_k w_k with w_k = d_k / t_k is
// rewritten over the common denominator prod_k t_k, so one IEEE division
// remains (the t_k are >= eps^2 and products of two or three of them stay in
// FP64's range); rounding differs from the reference's by a few ulps.

template <typename T>
__device__ __forceinline__ T rcp(T x) {
  if constexpr (sizeof(T) == 4) return __builtin_amdgcn_rcpf(x);
  else return T(1) / x;
}

// (c1 q1 / t1 + c2 q2 / t2) / (c1 / t1 + c2 / t2)
template <typename T>
__device__ __forceinline__ T blend2(T c1, T t1, T q1, T c2, T t2, T q2) {
  if constexpr (sizeof(T) == 4) {
    const T w1 = c1 * rcp(t1), w2 = c2 * rcp(t2);
    return (w1 * q1 + w2 * q2) * rcp(w1 + w2);
  } else {
    const T a1 = c1 * t2, a2 = c2 * t1;
    return (a1 * q1 + a2 * q2) / (a1 + a2);
  }
}

// (c1 q1 / t1 + c2 q2 / t2 + c3 q3 / t3) / (c1 / t1 + c2 / t2 + c3 / t3)
template <typename T>
__device__ __forceinline__ T blend3(T c1, T t1, T q1, T c2, T t2, T q2, T c3, T t3, T q3) {
  if constexpr (sizeof(T) == 4) {
    const T w1 = c1 * rcp(t1), w2 = c2 * rcp(t2), w3 = c3 * rcp(t3);
    return (w1 * q1 + w2 * q2 + w3 * q3) * rcp(w1 + w2 + w3);
  } else {
    const T a1 = c1 * (t2 * t3), a2 = c2 * (t1 * t3), a3 = c3 * (t1 * t2);
    return (a1 * q1 + a2 * q2 + a3 * q3) / (a1 + a2 + a3);
  }
}

template <typename T>
__device__ __forceinline__ T weno3_left(T qm, T q0, T qp) {  // weno.py:297-320
  const T eps = T(1e-8);
  const T qi1 = T(-0.5) * qm + T(1.5) * q0;
  const T qi2 = T(0.5) * (q0 + qp);
  const T b1 = (q0 - qm) * (q0 - qm), b2 = (qp - q0) * (qp - q0);
  const T t1 = b1 + eps, t2 = b2 + eps;
  // w1 = (1/3) / t1^2, w2 = (2/3) / t2^2
  return blend2(T(1.0 / 3.0), t1 * t1, qi1, T(2.0 / 3.0), t2 * t2, qi2);
}

template <typename T>
__device__ __forceinline__ T weno3_right(T q0, T qp, T qpp) {  // weno.py:413-435
  const T eps = T(1e-8);
  const T qi1 = T(0.5) * (q0 + qp);
  const T qi2 = T(1.5) * qp - T(0.5) * qpp;
  const T b1 = (qp - q0) * (qp - q0), b2 = (qpp - qp) * (qpp - qp);
  const T t1 = b1 + eps, t2 = b2 + eps;
  return blend2(T(2.0 / 3.0), t1 * t1, qi1, T(1.0 / 3.0), t2 * t2, qi2);
}

// WENO-Z weights d_k (1 + tau / (b_k + eps)) = d_k (b_k + eps + tau) / (b_k + eps).
template <typename T>
__device__ __forceinline__ T wenoz3_left(T qm, T q0, T qp) {  // weno.py:323-347
  const T eps = T(1e-14);
  const T qi1 = T(-0.5) * qm + T(1.5) * q0;
  const T qi2 = T(0.5) * (q0 + qp);
  const T b1 = (q0 - qm) * (q0 - qm), b2 = (qp - q0) * (qp - q0);
  const T tau = fabs(b2 - b1);
  if constexpr (sizeof(T) == 4) {
    const T w1 = T(1.0 / 3.0) * (T(1) + tau * rcp(b1 + eps));
    const T w2 = T(2.0 / 3.0) * (T(1) + tau * rcp(b2 + eps));
    return (w1 * qi1 + w2 * qi2) * rcp(w1 + w2);
  } else {
    const T t1 = b1 + eps, t2 = b2 + eps;
    return blend2(T(1.0 / 3.0) * (t1 + tau), t1, qi1, T(2.0 / 3.0) * (t2 + tau), t2, qi2);
  }
}

template <typename T>
__device__ __forceinline__ T wenoz3_right(T q0, T qp, T qpp) {  // weno.py:438-459
  const T eps = T(1e-14);
  const T qi1 = T(0.5) * (q0 + qp);
  const T qi2 = T(1.5) * qp - T(0.5) * qpp;
  const T b1 = (qp - q0) * (qp - q0), b2 = (qpp - qp) * (qpp - qp);
  const T tau = fabs(b2 - b1);
  if constexpr (sizeof(T) == 4) {
    const T w1 = T(2.0 / 3.0) * (T(1) + tau * rcp(b1 + eps));
    const T w2 = T(1.0 / 3.0) * (T(1) + tau * rcp(b2 + eps));
    return (w1 * qi1 + w2 * qi2) * rcp(w1 + w2);
  } else {
    const T t1 = b1 + eps, t2 = b2 + eps;
    return blend2(T(2.0 / 3.0) * (t1 + tau), t1, qi1, T(1.0 / 3.0) * (t2 + tau), t2, qi2);
  }
}

// WENO5 on the upwind-ordered stencil (a, b, c, d, e) = (qmm, qm, q0, qp, qpp)
// for positive flow and (qppp, qpp, qp, q0, qm) for negative flow: the
// right-biased reference formula (weno.py:462-491) is the left-biased one
// (weno.py:350-376) on the mirrored stencil, so one evaluation serves both.
//
// The face value is c + S with S a function of the four differences d1 = b - a,
// d2 = c - b, d3 = d - c, d4 = e - d alone:
//   candidates  - c : 5/6 d2 - 1/3 d1,  1/6 d2 + 1/3 d3,  2/3 d3 - 1/6 d4
//   indicators / k1 : s^2 + 3/13 r^2 (k1 = 13/12, k2 = 1/4) with
//                     s = d2 - d1, r = 2 d2 + s;  s = d3 - d2, r = d2 + d3;
//                     s = d4 - d3, r = s - 2 d3
// (the weights are ratios, so k1 divides out with eps / k1).  A difference is
// shared by the four faces around it and the mirrored stencil only reverses
// them, so a face costs ~55 issue slots instead of ~69 from five values.
// S is odd: the mirrored (negative) flow has S(-d) = -S(d).
template <typename T, bool Z>
__device__ __forceinline__ T weno5_delta(T d1, T d2, T d3, T d4) {
  const T p1 = T(5.0 / 6.0) * d2 - T(1.0 / 3.0) * d1;
  const T p2 = T(1.0 / 6.0) * d2 + T(1.0 / 3.0) * d3;
  const T p3 = T(2.0 / 3.0) * d3 - T(1.0 / 6.0) * d4;
  const T s1 = d2 - d1, r1 = T(2) * d2 + s1;  // a - 4 b + 3 c
  const T s2 = d3 - d2, r2 = d2 + d3;         // d - b
  const T s3 = d4 - d3, r3 = s3 - T(2) * d3;  // 3 c - 4 d + e
  const T k = T(3.0 / 13.0);
  if constexpr (!Z) {  // Jiang-Shu weights d_k / (b_k + eps)^2, eps 1e-8
    const T eps = T(1e-8 * 12.0 / 13.0);
    const T t1 = s1 * s1 + ((k * r1) * r1 + eps), t2 = s2 * s2 + ((k * r2) * r2 + eps),
            t3 = s3 * s3 + ((k * r3) * r3 + eps);
    return blend3(T(0.1), t1 * t1, p1, T(0.6), t2 * t2, p2, T(0.3), t3 * t3, p3);
  } else {  // WENO-Z (Borges et al. 2008), weno.py:379-410, eps 1e-16
    const T eps = T(1e-16 * 12.0 / 13.0);
    const T b1 = s1 * s1 + (k * r1) * r1, b2 = s2 * s2 + (k * r2) * r2,
            b3 = s3 * s3 + (k * r3) * r3;
    const T tau5 = fabs(b1 - b3);
    if constexpr (sizeof(T) == 4) {
      const T w1 = T(0.1) * (T(1) + tau5 * rcp(b1 + eps));
      const T w2 = T(0.6) * (T(1) + tau5 * rcp(b2 + eps));
      const T w3 = T(0.3) * (T(1) + tau5 * rcp(b3 + eps));
      return (w1 * p1 + w2 * p2 + w3 * p3) * rcp(w1 + w2 + w3);
    } else {
      const T t1 = b1 + eps, t2 = b2 + eps, t3 = b3 + eps;
      return blend3(T(0.1) * (t1 + tau5), t1, p1, T(0.6) * (t2 + tau5), t2, p2,
                    T(0.3) * (t3 + tau5), t3, p3);
    }
  }
}
template <typename T, bool Z>
__device__ __forceinline__ T weno5_upwind(T a, T b, T c, T d, T e) {
  return c + weno5_delta<T, Z>(b - a, c - b, d - c, e - d);
}
// The 3-point schemes' face value less c, from d2 = c - b and d3 = d - c (also
// odd).
template <typename T, bool Z>
__device__ __forceinline__ T weno3_delta(T d2, T d3) {
  const T b1 = d2 * d2, b2 = d3 * d3;
  if constexpr (!Z) {  // weno.py:297-320
    const T t1 = b1 + T(1e-8), t2 = b2 + T(1e-8);
    return T(0.5) * blend2(T(1.0 / 3.0), t1 * t1, d2, T(2.0 / 3.0), t2 * t2, d3);
  } else {  // weno.py:323-347
    const T t1 = b1 + T(1e-14), t2 = b2 + T(1e-14), tau = fabs(b2 - b1);
    if constexpr (sizeof(T) == 4) {
      const T w1 = T(1.0 / 3.0) * (T(1) + tau * rcp(t1)), w2 = T(2.0 / 3.0) * (T(1) + tau * rcp(t2));
      return T(0.5) * ((w1 * d2 + w2 * d3) * rcp(w1 + w2));
    } else {
      return T(0.5) * blend2(T(1.0 / 3.0) * (t1 + tau), t1, d2, T(2.0 / 3.0) * (t2 + tau), t2, d3);
    }
  }
}

template <typename T, int L>
__device__ __forceinline__ T limiter(T r) {  // advection/limiters.py:34-123
  if constexpr (L == kMinmod) return fmax(T(0), fmin(T(1), r));
  if constexpr (L == kVanLeer) {
    const T ra = fabs(r);
    return (r + ra) / (T(1) + ra);
  }
  if constexpr (L == kSuperbee) return fmax(T(0), fmax(fmin(T(2) * r, T(1)), fmin(r, T(2))));
  if constexpr (L == kMC) return fmax(T(0), fmin(fmin((T(1) + r) / T(2), T(2) * r), T(2)));
  return T(0);
}

// Face value at the face between cells i and i+1 along one direction.
// s[k * st] is h[i + k] for k in [-2, 3]; ``fi`` is the face index and ``n``
// the array length along the direction; only faces 1..n-3 are evaluated
// (the ones the tendency reads, advection.py:410-417).
template <typename T, int M, int L>
__device__ __forceinline__ T face_value(const T* s, int st, int fi, int n, bool pos) {
  const T h0 = s[0], h1 = s[st];
  if constexpr (M == kNaive) return T(0.5) * (h0 + h1);
  if constexpr (M == kUpwind1) return pos ? h0 : h1;
  const T hm1 = s[-st], h2 = s[2 * st];
  if constexpr (M == kUpwind2)  // reconstruction.py:636-657
    return pos ? T(1.5) * h0 - T(0.5) * hm1 : T(1.5) * h1 - T(0.5) * h2;
  if constexpr (M == kUpwind3)  // reconstruction.py:682-711
    return pos ? T(-1.0 / 6.0) * hm1 + T(5.0 / 6.0) * h0 + T(1.0 / 3.0) * h1
               : T(1.0 / 3.0) * h0 + T(5.0 / 6.0) * h1 - T(1.0 / 6.0) * h2;
  if constexpr (M == kWeno3)  // reconstruction.py:744-764
    return pos ? weno3_left(hm1, h0, h1) : weno3_right(h0, h1, h2);
  if constexpr (M == kWenoZ3)  // reconstruction.py:788-808
    return pos ? wenoz3_left(hm1, h0, h1) : wenoz3_right(h0, h1, h2);
  if constexpr (M == kWeno5 || M == kWenoZ5) {  // reconstruction.py:832-864 / 900-932
    constexpr bool Z = (M == kWenoZ5);
    if (pos) {
      if (fi == 1) return Z ? wenoz3_left(hm1, h0, h1) : weno3_left(hm1, h0, h1);
      return weno5_upwind<T, Z>(s[-2 * st], hm1, h0, h1, h2);
    }
    if (fi == n - 3) return Z ? wenoz3_right(h0, h1, h2) : weno3_right(h0, h1, h2);
    return weno5_upwind<T, Z>(s[3 * st], h2, h1, h0, hm1);
  }
  if constexpr (M == kTvd) {  // reconstruction.py:1000-1050, _TVD_EPS = 1e-8
    const T eps = T(1e-8);
    if (pos) {
      const T dfwd = h1 - h0, dbwd = h0 - hm1;
      return h0 + T(0.5) * limiter<T, L>(dbwd / (dfwd + eps)) * dfwd;
    }
    const T dneg = h0 - h1, dneg2 = h1 - h2;
    return h1 + T(0.5) * limiter<T, L>(dneg2 / (dneg + eps)) * dneg;
  }
  return T(0);
}

// Masked dispatch (flux.py:231-250): the upwind cell's tier picks the
// reconstruction {2: upwind1, 4: the 3-point scheme, 6: the 5-point scheme};
// tier 0 (land / no stencil) gives a zero flux.
template <typename T, int M, int L, bool MASKED>
__device__ __forceinline__ T face_flux(const T* s, int st, int fi, int n, T vel, int tier) {
  const bool pos = vel >= T(0);
  if constexpr (!MASKED) {
    return face_value<T, M, L>(s, st, fi, n, pos) * vel;
  } else {
    constexpr int cap = (M == kWeno5 || M == kWenoZ5) ? 6 : 4;
    constexpr int M4 = (M == kWenoZ5) ? kWenoZ3 : (M == kTvd ? kTvd : kWeno3);
    const int t = tier < cap ? tier : cap;
    if (t == 2) return face_value<T, kUpwind1, L>(s, st, fi, n, pos) * vel;
    if (t == 4) return face_value<T, M4, L>(s, st, fi, n, pos) * vel;
    if (t == 6) return face_value<T, M, L>(s, st, fi, n, pos) * vel;
    return T(0);
  }
}


// Optional fused Runge-Kutta stage: with hn set the kernel writes
// a hn + b h + cdt L(h) in place of L(h) (out may alias hn, not h).
template <typename T>
struct StageCoef {
  const T* hn = nullptr;
  double a = 0.0, b = 0.0, cdt = 0.0;
  // Periodic stages: the ghost width, and whether the output's ghosts are
  // written too (advection_kernel).
  int ng = 0, images = 0;
};

// Face value of the schemes of up to three points from the stencil mirrored to
// the upwind side of the face: (hm1, h0, h1) = h[i - 1], h[i], h[i + 1] for flow
// towards +x through the face between cells i and i+1, h[i + 2], h[i + 1], h[i]
// for flow towards -x.  Every scheme's negative-flow formula is its positive-flow
// formula on the mirrored stencil (weno.py:413-459 against :297-347,
// reconstruction.py:636-1050), so one branch-free evaluation serves both signs.
template <typename T, int M, int L>
__device__ __forceinline__ T upwind_value(T hm1, T h0, T h1) {
  if constexpr (M == kNaive) return T(0.5) * (h0 + h1);
  if constexpr (M == kUpwind1) return h0;
  if constexpr (M == kUpwind2) return T(1.5) * h0 - T(0.5) * hm1;
  if constexpr (M == kUpwind3)
    return T(-1.0 / 6.0) * hm1 + T(5.0 / 6.0) * h0 + T(1.0 / 3.0) * h1;
  if constexpr (M == kWeno3) return weno3_left(hm1, h0, h1);
  if constexpr (M == kWenoZ3) return wenoz3_left(hm1, h0, h1);
  if constexpr (M == kTvd) {
    const T eps = T(1e-8);
    const T dfwd = h1 - h0, dbwd = h0 - hm1;
    return h0 + T(0.5) * limiter<T, L>(dbwd / (dfwd + eps)) * dfwd;
  }
  return T(0);
}

// The masked tier dispatch of face_flux on the mirrored stencil.
template <typename T, int M, int L, bool MASKED>
__device__ __forceinline__ T upwind_face(T hm1, T h0, T h1, int tier) {
  if constexpr (!MASKED) {
    return upwind_value<T, M, L>(hm1, h0, h1);
  } else {
    constexpr int M4 = M == kTvd ? kTvd : kWeno3;
    if (tier == 2) return h0;
    if (tier >= 4) return upwind_value<T, M4, L>(hm1, h0, h1);
    return T(0);
  }
}

// WENO5 / WENO-Z5 flux through the face between values h0 and h1, from the
// differences around it (dk between cells k and k + 1 of the face's cell 0):
// the upwind cell's value plus or minus the oriented weno5_delta; the masked
// tier dispatch of face_flux.  ``near``: the face next to the array edge on the
// upwind side (face 1 for positive, n - 3 for negative flow), where these schemes
// fall back to the 3-point ones.
template <typename T, bool Z, bool MASKED>
__device__ __forceinline__ T weno5_flux(T h0, T h1, T dm2, T dm1, T d0, T d1, T d2, T vel,
                                        bool near, int tier) {
  const bool pos = vel >= T(0);
  const T a1 = pos ? dm2 : d2, a2 = pos ? dm1 : d1, a4 = pos ? d1 : dm1;
  // (a map may hold the largest stencil that fits, so 6 and above is 6)
  const bool five = !MASKED || tier >= 6, three = tier == 4;
  T sd = T(0);
  if (five) {
    if (near) sd = weno3_delta<T, Z>(a2, d0);
    else sd = weno5_delta<T, Z>(a1, a2, d0, a4);
  } else if (three) {
    sd = weno3_delta<T, Z>(a2, d0);
  }
  const T f = ((pos ? h0 : h1) + (pos ? sd : -sd)) * vel;
  return (five || three || tier == 2) ? f : T(0);
}

// One wavefront per tile of 58 output columns (lanes 3..60; three halo lanes
// each side) x R rows.  Each lane keeps its column of h on rows
// j0-3 .. j0+R+2 in registers; the x stencils come from DPP lane
// shifts, the y stencils from neighbouring registers.  Each lane evaluates
// the east face of its cell (the west face is the east face of the lane
// beside it) and the north faces of its column, so every face flux is
// reconstructed once; no LDS, no barriers, no integer division per cell.
// Grids up to 512^2 take tiles of 2 rows: more wavefronts for the chip, a
// shorter chain of loads and arithmetic per wavefront.
//
// Bound by issue slots and by the loads' latency (2048^2 FP64 0.54 of the VALU's
// issue peak and 0.47 of the bandwidth, FP32 0.68 and 0.38; masked 0.42 / 0.39 and
// 0.54 / 0.35), so: differences instead of values (weno5_delta); every array of the tile
// requested before the first flux (a stage's output may alias its h_n, so the
// compiler does not move those loads up itself); and a tile away from every
// edge (INNER: all but the outermost ring) runs without the clamps, zero
// fills, fallbacks and ring tests of the others.  One Advection2D call, us,
// before and now, FP64 / FP32 (the prefetch costs FP64 one wavefront in four a
// SIMD, 3 instead of 4, and is still worth it):
//   weno5 2048^2          48.5 -> 37.2 / 30.4 -> 23.5
//   weno5 3000^2         114.5 -> 76.7 / 48.4 -> 40.6
//   weno5 masked 3000^2  144.5 -> 106.9 / 66.4 -> 48.3
//   van_leer 3000^2       65.3 -> 58.4 / 34.6 -> 32.7
//
// Periodic stages (ng > 0: the ghost width): h is read through the index map
// of enforce_periodic (a ghost cell is its doubly wrapped interior cell), so
// the caller fills no ghosts between stages; only interior cells are written,
// with ``images`` also the ghost cells that copy them.
constexpr int kAdvRows = 8, kAdvShortRows = 2, kAdvCols = 58;
constexpr int64_t kAdvShortMaxCells = 514 * 514;

template <typename T>
__device__ __forceinline__ T adv_e(T v) {
  return dpp_move<0x130>(v);  // wave_shl 1: value of lane + 1, 0 in lane 63
}
template <typename T>
__device__ __forceinline__ T adv_w(T v) {
  return dpp_move<0x138>(v);  // wave_shr 1: value of lane - 1, 0 in lane 0
}
// Index of the cell that cell k of n holds after the periodic fill.
__device__ __forceinline__ int adv_wrap(int k, int n, int ng) {
  return k < ng ? k + (n - 2 * ng) : (k >= n - ng ? k - (n - 2 * ng) : k);
}

template <typename T>
struct AdvArgs {
  const T *h, *u, *v;
  T* out;
  const uint8_t *tier_x, *tier_y, *mh;
  int ny, nx;
  T idx, idy;
  int tiles_x, ntiles;
  const T* hn;
  T ca, cb, ccdt;
  int ng, images;
};

// INNER: every cell, face and stencil of the tile lies inside the array, away
// from the edge fallbacks, the output ring and the periodic ghosts and images.
template <typename T, int M, int L, bool MASKED, int R, bool INNER>
__device__ __forceinline__ void advection_tile(const AdvArgs<T>& a, int i0, int j0, int lane) {
  constexpr int HR = R + 6;
  constexpr bool W5 = M == kWeno5 || M == kWenoZ5, Z = M == kWenoZ5;
  const int ny = a.ny, nx = a.nx, ng = INNER ? 0 : a.ng;
  const int gi = i0 - 3 + lane;
  const bool colin = INNER || (gi >= 0 && gi < nx);
  const unsigned gic = INNER ? (unsigned)gi : (unsigned)min(max(gi, 0), nx - 1);
  const unsigned gih = (unsigned)(ng > 0 ? adv_wrap((int)gic, nx, ng) : (int)gic);
  auto row = [&](int gj) -> int64_t {
    return (int64_t)(INNER ? gj : min(max(gj, 0), ny - 1)) * nx;
  };
  // h on rows j0-3+r (zero outside the array), v on rows j0-1 .. j0+R-1 (the
  // faces between rows j0-1+t and j0+t), u on the output rows
  T hr[HR], vr[R + 1], ur[R], hs[R];
  int tyr[MASKED ? R + 2 : 1], txr[MASKED ? R : 1], mr[R];
#pragma unroll
  for (int r = 0; r < HR; ++r) {
    if constexpr (INNER) {
      hr[r] = (a.h + row(j0 - 3 + r))[gih];
    } else {
      const int gj = min(max(j0 - 3 + r, 0), ny - 1);
      hr[r] = (a.h + (int64_t)(ng > 0 ? adv_wrap(gj, ny, ng) : gj) * nx)[gih];
    }
  }
#pragma unroll
  for (int t = 0; t <= R; ++t) vr[t] = (a.v + row(j0 - 1 + t))[gic];
#pragma unroll
  for (int t = 0; t < R; ++t) ur[t] = (a.u + row(j0 + t))[gic];
  if constexpr (MASKED) {
#pragma unroll
    for (int t = 0; t < R + 2; ++t) tyr[t] = (a.tier_y + row(j0 - 1 + t))[gic];
#pragma unroll
    for (int t = 0; t < R; ++t) txr[t] = (a.tier_x + row(j0 + t))[gic];
  }
#pragma unroll
  for (int t = 0; t < R; ++t) {
    mr[t] = a.mh ? (a.mh + row(j0 + t))[gic] : 1;
    hs[t] = a.hn ? (a.hn + row(j0 + t))[gic] : T(0);
  }
  if constexpr (!INNER) {
#pragma unroll
    for (int r = 0; r < HR; ++r) {
      const int gj = j0 - 3 + r;
      if (!colin || gj < 0 || gj >= ny) hr[r] = T(0);
    }
  }
  // (W5) differences of neighbouring rows, shared by the faces around them
  T dy_[W5 ? HR - 1 : 1];
  if constexpr (W5) {
#pragma unroll
    for (int r = 0; r < HR - 1; ++r) dy_[r] = hr[r + 1] - hr[r];
  }
  // North faces fj = j0-1+t (between rows j0-1+t and j0+t), t = 0 .. R.
  T fn[R + 1];
#pragma unroll
  for (int t = 0; t <= R; ++t) {
    const int r = t + 2, fj = j0 - 1 + t;
    const T vel = vr[t];
    const bool pos = vel >= T(0);
    int tier = 0;
    if constexpr (MASKED) {
      tier = pos ? tyr[t] : tyr[t + 1];
    }
    const bool near = !INNER && (pos ? fj == 1 : fj == ny - 3);
    T f;
    if constexpr (W5) {
      f = weno5_flux<T, Z, MASKED>(hr[r], hr[r + 1], dy_[r - 2], dy_[r - 1], dy_[r], dy_[r + 1],
                                   dy_[r + 2], vel, near, tier);
    } else {
      f = upwind_face<T, M, L, MASKED>(pos ? hr[r - 1] : hr[r + 2], pos ? hr[r] : hr[r + 1],
                                       pos ? hr[r + 1] : hr[r], tier) * vel;
    }
    fn[t] = INNER || (colin && gi >= 2 && gi <= nx - 3 && fj >= 1 && fj <= ny - 3) ? f : T(0);
  }
  const bool lout = colin && lane >= 3 && lane <= 60 && (ng == 0 || (gi >= ng && gi < nx - ng));
#pragma unroll
  for (int t = 0; t < R; ++t) {
    const int r = t + 3, gj = j0 + t;
    // East face fi = gi of this row (between columns gi and gi+1).
    const T hc = hr[r];
    const T e1 = adv_e(hc);
    const T vel = ur[t];
    const bool pos = vel >= T(0);
    int tier = 0;
    if constexpr (MASKED) {
      const int txe = __builtin_amdgcn_mov_dpp(txr[t], 0x130, 0xf, 0xf, true);  // lane + 1
      tier = pos ? txr[t] : txe;
    }
    const bool near = !INNER && (pos ? gi == 1 : gi == nx - 3);
    T fe;
    if constexpr (W5) {
      const T d0 = e1 - hc, dm1 = adv_w(d0), dm2 = adv_w(dm1), d1 = adv_e(d0), d2 = adv_e(d1);
      fe = weno5_flux<T, Z, MASKED>(hc, e1, dm2, dm1, d0, d1, d2, vel, near, tier);
    } else {
      const T e2 = adv_e(e1), w1 = adv_w(hc);
      fe = upwind_face<T, M, L, MASKED>(pos ? w1 : e2, pos ? hc : e1, pos ? e1 : hc, tier) * vel;
    }
    if constexpr (!INNER)
      fe = colin && gj >= 2 && gj <= ny - 3 && gi >= 1 && gi <= nx - 3 ? fe : T(0);
    const T fw = adv_w(fe);
    if (lout && (INNER || (gj < ny && (ng == 0 || (gj >= ng && gj < ny - ng))))) {
      T res = T(0);
      if (INNER || (gj >= 2 && gj <= ny - 3 && gi >= 2 && gi <= nx - 3))
        res = -((fe - fw) * a.idx + (fn[t + 1] - fn[t]) * a.idy);
      if (a.mh) res = res * (T)(mr[t] ? 1 : 0);
      if (a.hn) res = a.ca * hs[t] + a.cb * hc + a.ccdt * res;
      T* o = a.out + (int64_t)gj * nx;
      o[gi] = res;
      if (!INNER && a.images) {  // the ghost cells this cell fills
        const int pi = nx - 2 * ng, pj = ny - 2 * ng;
        const bool xe = gi < 2 * ng, xw = gi >= nx - 2 * ng;  // image east / west
        if (xe) o[gi + pi] = res;
        if (xw) o[gi - pi] = res;
        if (gj < 2 * ng) {
          T* q = o + (int64_t)pj * nx;
          q[gi] = res;
          if (xe) q[gi + pi] = res;
          if (xw) q[gi - pi] = res;
        }
        if (gj >= ny - 2 * ng) {
          T* q = o - (int64_t)pj * nx;
          q[gi] = res;
          if (xe) q[gi + pi] = res;
          if (xw) q[gi - pi] = res;
        }
      }
    }
  }
}

template <typename T, int M, int L, bool MASKED, int R>
__global__ __launch_bounds__(256) void advection_kernel(AdvArgs<T> a) {
  const int lane = threadIdx.x & 63;
  const int tile =
      __builtin_amdgcn_readfirstlane(xcd_swizzle(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6));
  if (tile >= a.ntiles) return;  // whole wavefront (no block-level barrier below)
  const int tyi = tile / a.tiles_x;
  const int i0 = (tile - tyi * a.tiles_x) * kAdvCols, j0 = tyi * R;
  const int mg = 2 * a.ng;
  const bool inner = i0 - 3 >= mg && i0 + 61 <= a.nx - mg && j0 - 3 >= mg && j0 + R + 3 <= a.ny - mg;
  if (inner) advection_tile<T, M, L, MASKED, R, true>(a, i0, j0, lane);
  else advection_tile<T, M, L, MASKED, R, false>(a, i0, j0, lane);
}

template <typename T, int M, int L, bool MASKED>
static void launch_adv(const T* h, const T* u, const T* v, T* out, const uint8_t* tx_,
                       const uint8_t* ty_, const uint8_t* mh, int ny, int nx, double dx,
                       double dy, const StageCoef<T>& sc, hipStream_t s) {
  const bool short_tiles = (int64_t)ny * nx <= kAdvShortMaxCells;
  const int rows = short_tiles ? kAdvShortRows : kAdvRows;
  const int tiles_x = cdiv(nx, kAdvCols), tiles_y = cdiv(ny, rows);
  const int ntiles = tiles_x * tiles_y;
  const AdvArgs<T> a{h,  u,  v,  out, tx_, ty_, mh, ny, nx, (T)(1.0 / dx), (T)(1.0 / dy), tiles_x,
                     ntiles, sc.hn, (T)sc.a, (T)sc.b, (T)sc.cdt, sc.ng, sc.images};
  const dim3 grid(cdiv(ntiles, 4)), block(256);
  if (short_tiles)
    hipLaunchKernelGGL((advection_kernel<T, M, L, MASKED, kAdvShortRows>), grid, block, 0, s, a);
  else
    hipLaunchKernelGGL((advection_kernel<T, M, L, MASKED, kAdvRows>), grid, block, 0, s, a);
}

template <typename T, bool MASKED>
static int dispatch_adv(int method, int lim, const T* h, const T* u, const T* v, T* out,
                        const uint8_t* tx_, const uint8_t* ty_, const uint8_t* mh, int ny,
                        int nx, double dx, double dy, const StageCoef<T>& sc, hipStream_t s) {
#define FVX_ADV(M, L) \
  launch_adv<T, M, L, MASKED>(h, u, v, out, tx_, ty_, mh, ny, nx, dx, dy, sc, s)
  if constexpr (MASKED) {
    switch (method) {
      case kWeno3: FVX_ADV(kWeno3, 0); break;
      case kWeno5: FVX_ADV(kWeno5, 0); break;
      case kWenoZ5: FVX_ADV(kWenoZ5, 0); break;
      case kTvd:
        switch (lim) {
          case kMinmod: FVX_ADV(kTvd, kMinmod); break;
          case kVanLeer: FVX_ADV(kTvd, kVanLeer); break;
          case kSuperbee: FVX_ADV(kTvd, kSuperbee); break;
          case kMC: FVX_ADV(kTvd, kMC); break;
          default: set_error("unknown limiter %d", lim); return kInvalidArgument;
        }
        break;
      default:
        set_error("method %d does not support mask-based stencil dispatch", method);
        return kInvalidArgument;
    }
  } else {
    switch (method) {
      case kNaive: FVX_ADV(kNaive, 0); break;
      case kUpwind1: FVX_ADV(kUpwind1, 0); break;
      case kUpwind2: FVX_ADV(kUpwind2, 0); break;
      case kUpwind3: FVX_ADV(kUpwind3, 0); break;
      case kWeno3: FVX_ADV(kWeno3, 0); break;
      case kWenoZ3: FVX_ADV(kWenoZ3, 0); break;
      case kWeno5: FVX_ADV(kWeno5, 0); break;
      case kWenoZ5: FVX_ADV(kWenoZ5, 0); break;
      case kTvd:
        switch (lim) {
          case kMinmod: FVX_ADV(kTvd, kMinmod); break;
          case kVanLeer: FVX_ADV(kTvd, kVanLeer); break;
          case kSuperbee: FVX_ADV(kTvd, kSuperbee); break;
          case kMC: FVX_ADV(kTvd, kMC); break;
          default: set_error("unknown limiter %d", lim); return kInvalidArgument;
        }
        break;
      default: set_error("unknown advection method %d", method); return kInvalidArgument;
    }
  }
#undef FVX_ADV
  FVX_LAUNCH_CHECK();
  return kOk;
}

template <typename T>
int advection(int method, int lim, const T* h, const T* u, const T* v, T* out,
              const uint8_t* tier_x, const uint8_t* tier_y, const uint8_t* mh, int ny, int nx,
              double dx, double dy, hipStream_t s, const StageCoef<T>& sc = StageCoef<T>()) {
  FVX_CHECK_ARG(h && u && v && out, "null field pointer");
  FVX_CHECK_ARG(ny >= 5 && nx >= 5, "array too small (%d x %d); need >= 5 x 5", ny, nx);
  FVX_CHECK_ARG(dx > 0 && dy > 0, "grid spacing must be positive");
  FVX_CHECK_ARG((tier_x == nullptr) == (tier_y == nullptr), "tier_x and tier_y go together");
  FVX_CHECK_ARG(out != h, "out must not alias h (neighbouring tiles still read it)");
  if (tier_x)
    return dispatch_adv<T, true>(method, lim, h, u, v, out, tier_x, tier_y, mh, ny, nx, dx, dy,
                                 sc, s);
  return dispatch_adv<T, false>(method, lim, h, u, v, out, nullptr, nullptr, mh, ny, nx, dx, dy,
                                sc, s);
}

// ---------------------------------------------------------------------------
// Face fluxes of one direction (Reconstruction2D.<method>_x / _y and the
// *_masked variants, reconstruction.py:582-1307): every face 1..n-2 along the
// direction on rows (columns) 1..m-2, zero ring.  Faces the tendency never
// reads fall back as the reference does: at the last face n-2 positive flow
// takes the 3-point scheme in place of the 5-point one and negative flow
// takes upwind1 (the value beyond the face) for every scheme but naive.
// One thread per face; its six stencil values are loaded into registers
// (zero beyond the array).
// ---------------------------------------------------------------------------
template <typename T, int M, int L, bool MASKED>
__device__ __forceinline__ T face_flux_any(const T* s, int fi, int n, T vel, int tier) {
  if (fi == n - 2 && M != kNaive) {
    const bool pos = vel >= T(0);
    if (!pos) {
      if (MASKED && tier < 2) return T(0);
      return s[1] * vel;
    }
    if constexpr (M == kWeno5 || M == kWenoZ5) {
      constexpr int M3 = (M == kWeno5) ? kWeno3 : kWenoZ3;
      if (MASKED && tier < 2) return T(0);
      if (MASKED && tier == 2) return s[0] * vel;
      return face_value<T, M3, L>(s, 1, fi, n, true) * vel;
    }
  }
  return face_flux<T, M, L, MASKED>(s, 1, fi, n, vel, tier);
}

template <typename T, int M, int L, bool MASKED, bool YDIR>
__global__ __launch_bounds__(256) void face_flux_kernel(const T* __restrict__ h,
                                                        const T* __restrict__ vel,
                                                        T* __restrict__ out,
                                                        const uint8_t* __restrict__ tier, int ny,
                                                        int nx) {
  const int i = blockIdx.x * 64 + (threadIdx.x & 63);
  const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (i >= nx || j >= ny) return;
  const int64_t c = (int64_t)j * nx + i;
  const int fi = YDIR ? j : i, n = YDIR ? ny : nx;
  const int oi = YDIR ? i : j, m = YDIR ? nx : ny;
  const int64_t st = YDIR ? nx : 1;
  T f = T(0);
  if (fi >= 1 && fi <= n - 2 && oi >= 1 && oi <= m - 2) {
    T w[6];
#pragma unroll
    for (int k = -2; k <= 3; ++k) {
      const int q = fi + k;
      w[k + 2] = (q >= 0 && q < n) ? h[c + k * st] : T(0);
    }
    const T v = vel[c];
    int t = 6;
    if constexpr (MASKED) t = (v >= T(0)) ? tier[c] : tier[c + st];
    f = face_flux_any<T, M, L, MASKED>(w + 2, fi, n, v, t);
  }
  out[c] = f;
}

template <typename T, int M, int L, bool MASKED>
static void launch_face_flux(int dir, const T* h, const T* vel, T* out, const uint8_t* tier,
                             int ny, int nx, hipStream_t s) {
  const dim3 g(cdiv(nx, 64), cdiv(ny, 4));
  if (dir == 0)
    hipLaunchKernelGGL((face_flux_kernel<T, M, L, MASKED, false>), g, dim3(256), 0, s, h, vel,
                       out, tier, ny, nx);
  else
    hipLaunchKernelGGL((face_flux_kernel<T, M, L, MASKED, true>), g, dim3(256), 0, s, h, vel, out,
                       tier, ny, nx);
}

template <typename T>
int face_flux_call(int method, int lim, int dir, const T* h, const T* vel, T* out,
                   const uint8_t* tier, int ny, int nx, hipStream_t s) {
  FVX_CHECK_ARG(h && vel && out, "null field pointer");
  FVX_CHECK_ARG(dir == 0 || dir == 1, "dir must be 0 (x, east faces) or 1 (y, north faces)");
  FVX_CHECK_ARG(ny >= 3 && nx >= 3, "array too small (%d x %d)", ny, nx);
  FVX_CHECK_ARG(lim >= 0 && lim <= 3, "unknown limiter %d", lim);
#define FVX_FF(M, L)                                                                 \
  (tier ? launch_face_flux<T, M, L, true>(dir, h, vel, out, tier, ny, nx, s)          \
        : launch_face_flux<T, M, L, false>(dir, h, vel, out, tier, ny, nx, s))
  if (tier) {
    FVX_CHECK_ARG(method == kWeno3 || method == kWeno5 || method == kWenoZ5 || method == kTvd,
                  "method %d does not support mask-based stencil dispatch", method);
  }
  switch (method) {
    case kNaive: launch_face_flux<T, kNaive, 0, false>(dir, h, vel, out, nullptr, ny, nx, s); break;
    case kUpwind1: launch_face_flux<T, kUpwind1, 0, false>(dir, h, vel, out, nullptr, ny, nx, s); break;
    case kUpwind2: launch_face_flux<T, kUpwind2, 0, false>(dir, h, vel, out, nullptr, ny, nx, s); break;
    case kUpwind3: launch_face_flux<T, kUpwind3, 0, false>(dir, h, vel, out, nullptr, ny, nx, s); break;
    case kWenoZ3: launch_face_flux<T, kWenoZ3, 0, false>(dir, h, vel, out, nullptr, ny, nx, s); break;
    case kWeno3: FVX_FF(kWeno3, 0); break;
    case kWeno5: FVX_FF(kWeno5, 0); break;
    case kWenoZ5: FVX_FF(kWenoZ5, 0); break;
    case kTvd:
      switch (lim) {
        case kMinmod: FVX_FF(kTvd, kMinmod); break;
        case kVanLeer: FVX_FF(kTvd, kVanLeer); break;
        case kSuperbee: FVX_FF(kTvd, kSuperbee); break;
        default: FVX_FF(kTvd, kMC); break;
      }
      break;
    default: set_error("unknown advection method %d", method); return kInvalidArgument;
  }
#undef FVX_FF
  FVX_LAUNCH_CHECK();
  return kOk;
}

// ---------------------------------------------------------------------------
// One rk3_ssp_step (timestepping/explicit_rk.py:74-121) of a doubly periodic
// tracer: per stage the periodic ghost fill of width ng (boundary.py:52-78,
// as the periodic advection tests do before each tendency) and the
// Advection2D tendency with the Shu-Osher combination, in one launch each:
// the stages read their input through the fill's index map, and the last one
// writes the result's ghosts.  Scratch: the two stage states y1, y2 (interior
// only).  Per step, FP64 WENO5: 38.7 us with the fills as launches of their own,
// now 17.1 at 256^2 (the three kernels take 16);
// 83 -> 47 at 1000^2, 104 -> 72 at 1500^2.
// ---------------------------------------------------------------------------

// Argument checks shared by both entry points (no device work).
template <typename T>
static int adv_rk3_check(const T* h, const T* u, const T* v, int ny, int nx, int ng, double dx,
                         double dy, double dt) {
  FVX_CHECK_ARG(h && u && v, "null field pointer");
  FVX_CHECK_ARG(ng >= 1 && ny >= 3 * ng && nx >= 3 * ng && ny >= 5 && nx >= 5,
                "ghost width %d too large for %d x %d", ng, ny, nx);
  FVX_CHECK_ARG(dx > 0 && dy > 0, "grid spacing must be positive");
  FVX_CHECK_ARG(std::isfinite(dt), "dt must be finite");
  return kOk;
}

// h -> res (which may be h).
template <typename T>
static int adv_rk3_enqueue(int method, int lim, const T* h, T* res, const T* u, const T* v,
                           const uint8_t* tier_x, const uint8_t* tier_y, const uint8_t* mh,
                           int ny, int nx, int ng, double dx, double dy, double dt, T* y1, T* y2,
                           hipStream_t s) {
  // Each stage is one advection launch with the Shu-Osher combination fused
  // (out = a h + b q + cdt L(q) on every interior cell, q the stage's input).
  auto stage = [&](const T* q, T* out, double a, double b, double cdt, int images) {
    StageCoef<T> sc;
    sc.hn = h;
    sc.a = a;
    sc.b = b;
    sc.cdt = cdt;
    sc.ng = ng;
    sc.images = images;
    return advection<T>(method, lim, q, u, v, out, tier_x, tier_y, mh, ny, nx, dx, dy, s, sc);
  };
  // y1 = h + dt L(h), y2 = 3/4 h + 1/4 y1 + 1/4 dt L(y1),
  // 1/3 h + 2/3 y2 + 2/3 dt L(y2) (the output may alias h: an interior cell is
  // read by the lane that writes it, a ghost cell is not read)
  if (int rc = stage(h, y1, 0.0, 1.0, dt, 0)) return rc;
  if (int rc = stage(y1, y2, 0.75, 0.25, 0.25 * dt, 0)) return rc;
  return stage(y2, res, 1.0 / 3.0, 2.0 / 3.0, 2.0 / 3.0 * dt, 1);
}

// Stage arrays of the allocating entry point: one buffer per device, grown
// with hipMalloc when a call needs more and kept until the process ends.
static std::mutex g_stage_mu;
static void* g_stage_buf[64] = {};
static size_t g_stage_bytes[64] = {};

template <typename T>
static int adv_rk3_step(int method, int lim, T* h, const T* u, const T* v,
                        const uint8_t* tier_x, const uint8_t* tier_y, const uint8_t* mh, int ny,
                        int nx, int ng, double dx, double dy, double dt, hipStream_t s) {
  if (int rc = adv_rk3_check<T>(h, u, v, ny, nx, ng, dx, dy, dt)) return rc;
  const size_t bytes = 2 * (size_t)ny * nx * sizeof(T);
  int dev = 0;
  FVX_HIP(hipGetDevice(&dev));
  FVX_CHECK_ARG(dev >= 0 && dev < 64, "device index %d out of range", dev);
  T* buf = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_stage_mu);
    if (g_stage_bytes[dev] < bytes) {
      // earlier work on any stream may still use the old buffer
      FVX_HIP(hipDeviceSynchronize());
      if (g_stage_buf[dev]) FVX_HIP(hipFree(g_stage_buf[dev]));
      g_stage_buf[dev] = nullptr;
      g_stage_bytes[dev] = 0;
      FVX_HIP(hipMalloc(&g_stage_buf[dev], bytes));
      g_stage_bytes[dev] = bytes;
    }
    buf = (T*)g_stage_buf[dev];
  }
  return adv_rk3_enqueue<T>(method, lim, h, h, u, v, tier_x, tier_y, mh, ny, nx, ng, dx, dy, dt,
                            buf, buf + (size_t)ny * nx, s);
}

// The allocation-free variant keeps the two stage arrays in ``scratch``, a
// device array of kAdvScratchBytes that every GPU holds until the process
// ends; calls on one GPU share it (overlapping calls on one GPU race).  Host
// code never uses the array's name as an address: the first call on each
// device looks its address up with hipGetSymbolAddress (device current) and
// keeps it per device.
constexpr size_t kAdvScratchBytes = size_t(32) << 20;
static __device__ __align__(256) unsigned char scratch[kAdvScratchBytes];
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[64] = {};

static int scratch_ptr(void** out) {
  int dev = 0;
  FVX_HIP(hipGetDevice(&dev));
  FVX_CHECK_ARG(dev >= 0 && dev < 64, "device index %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      set_error("hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
      return kHipError;
    }
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return kOk;
}

template <typename T>
static int adv_rk3_step_noalloc(int method, int lim, T* h, const T* u, const T* v,
                                const uint8_t* tier_x, const uint8_t* tier_y,
                                const uint8_t* mh, int ny, int nx, int ng, double dx, double dy,
                                double dt, hipStream_t s) {
  if (int rc = adv_rk3_check<T>(h, u, v, ny, nx, ng, dx, dy, dt)) return rc;
  const size_t bytes = 2 * (size_t)ny * nx * sizeof(T);
  FVX_CHECK_ARG(bytes <= kAdvScratchBytes,
                "%d x %d needs %zu bytes of stage scratch; the allocation-free step holds "
                "%zu (two arrays of at most %zu elements)",
                ny, nx, bytes, kAdvScratchBytes, kAdvScratchBytes / (2 * sizeof(T)));
  void* p = nullptr;
  if (int rc = scratch_ptr(&p)) return rc;
  T* y1 = (T*)p;
  return adv_rk3_enqueue<T>(method, lim, h, h, u, v, tier_x, tier_y, mh, ny, nx, ng, dx, dy, dt, y1,
                            y1 + (size_t)ny * nx, s);
}

}  // namespace fvx

extern "C" {
#define FVX_ADV_RK3(SUF, T)                                                                      \
  int fvx_advection_rk3_step_##SUF(int method, int limiter, T* h, const T* u, const T* v,        \
                                   const uint8_t* tier_x, const uint8_t* tier_y,                \
                                   const uint8_t* mask_h, int ny, int nx, int ng, double dx,    \
                                   double dy, double dt, void* stream) {                        \
    return fvx::adv_rk3_step<T>(method, limiter, h, u, v, tier_x, tier_y, mask_h, ny, nx, ng,   \
                                dx, dy, dt, (hipStream_t)stream);                               \
  }                                                                                              \
  int fvx_advection_rk3_step_noalloc_##SUF(int method, int limiter, T* h, const T* u,           \
                                           const T* v, const uint8_t* tier_x,                   \
                                           const uint8_t* tier_y, const uint8_t* mask_h,        \
                                           int ny, int nx, int ng, double dx, double dy,        \
                                           double dt, void* stream) {                           \
    return fvx::adv_rk3_step_noalloc<T>(method, limiter, h, u, v, tier_x, tier_y, mask_h, ny,   \
                                        nx, ng, dx, dy, dt, (hipStream_t)stream);               \
  }
FVX_ADV_RK3(f32, float)
FVX_ADV_RK3(f64, double)
#undef FVX_ADV_RK3

// The step from h into out (another array), with the caller's scratch of
// 2 ny nx elements: no allocation, no array shared with other calls.
#define FVX_ADV_RK3_INTO(SUF, T)                                                                 \
  int fvx_advection_rk3_step_into_##SUF(int method, int limiter, const T* h, T* out, const T* u, \
                                        const T* v, const uint8_t* tier_x,                       \
                                        const uint8_t* tier_y, const uint8_t* mask_h, int ny,    \
                                        int nx, int ng, double dx, double dy, double dt,         \
                                        T* work, void* stream) {                                 \
    if (int rc = fvx::adv_rk3_check<T>(h, u, v, ny, nx, ng, dx, dy, dt)) return rc;              \
    FVX_CHECK_ARG(out && work, "null field pointer");                                            \
    FVX_CHECK_ARG(out != h, "out must not alias h");                                             \
    return fvx::adv_rk3_enqueue<T>(method, limiter, h, out, u, v, tier_x, tier_y, mask_h, ny,    \
                                   nx, ng, dx, dy, dt, work, work + (size_t)ny * nx,             \
                                   (hipStream_t)stream);                                         \
  }
FVX_ADV_RK3_INTO(f32, float)
FVX_ADV_RK3_INTO(f64, double)
#undef FVX_ADV_RK3_INTO

int fvx_face_flux_f64(int method, int limiter, int dir, const double* h, const double* vel,
                      double* out, const uint8_t* tier, int ny, int nx, void* stream) {
  return fvx::face_flux_call<double>(method, limiter, dir, h, vel, out, tier, ny, nx,
                                     (hipStream_t)stream);
}
int fvx_face_flux_f32(int method, int limiter, int dir, const float* h, const float* vel,
                      float* out, const uint8_t* tier, int ny, int nx, void* stream) {
  return fvx::face_flux_call<float>(method, limiter, dir, h, vel, out, tier, ny, nx,
                                    (hipStream_t)stream);
}

#define FVX_ADV_STAGE(SUF, T)                                                                    \
  int fvx_advection_stage_##SUF(int method, int limiter, const T* hs, const T* u, const T* v,    \
                                const T* hn, T* out, const uint8_t* tier_x,                     \
                                const uint8_t* tier_y, const uint8_t* mask_h, int ny, int nx,   \
                                double dx, double dy, double a, double b, double cdt,           \
                                void* stream) {                                                 \
    FVX_CHECK_ARG(hn, "null hn");                                                               \
    fvx::StageCoef<T> sc;                                                                        \
    sc.hn = hn;                                                                                  \
    sc.a = a;                                                                                    \
    sc.b = b;                                                                                    \
    sc.cdt = cdt;                                                                                \
    return fvx::advection<T>(method, limiter, hs, u, v, out, tier_x, tier_y, mask_h, ny, nx, dx, \
                             dy, (hipStream_t)stream, sc);                                       \
  }
FVX_ADV_STAGE(f32, float)
FVX_ADV_STAGE(f64, double)
#undef FVX_ADV_STAGE

int fvx_advection2d_f64(int method, int limiter, const double* h, const double* u,
                        const double* v, double* out, const uint8_t* tier_x,
                        const uint8_t* tier_y, const uint8_t* mask_h, int ny, int nx,
                        double dx, double dy, void* stream) {
  return fvx::advection<double>(method, limiter, h, u, v, out, tier_x, tier_y, mask_h, ny, nx,
                                dx, dy, (hipStream_t)stream);
}
int fvx_advection2d_f32(int method, int limiter, const float* h, const float* u,
                        const float* v, float* out, const uint8_t* tier_x,
                        const uint8_t* tier_y, const uint8_t* mask_h, int ny, int nx,
                        double dx, double dy, void* stream) {
  return fvx::advection<float>(method, limiter, h, u, v, out, tier_x, tier_y, mask_h, ny, nx,
                               dx, dy, (hipStream_t)stream);
}
}
