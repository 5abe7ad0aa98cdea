// C-grid stencils: Difference2D / Divergence2D / Interpolation2D point ops,
// Diffusion2D (+ fluxes), fused BiharmonicDiffusion2D, the Arakawa Jacobian,
// masked_laplacian and the periodic ghost fill.
//
// All kernels are HBM-bandwidth bound; each output element is written once
// and each input element is read from HBM once (neighbour reuse comes from L1,
// registers and lane moves).  A wavefront covers 60 to 64 contiguous columns of
// one or several rows.

#include "fvx_common.hpp"

namespace fvx {

// Operator codes of the point-stencil family; the order is part of the C ABI
// (include/fvx.h, FVX_OP_*).
enum StencilOp : int {
  kDiffX_T2U = 0,   // difference.py:194  (h[j,i+1]-h[j,i])/dx        mask u
  kDiffY_T2V = 1,   // difference.py:215  (h[j+1,i]-h[j,i])/dy        mask v
  kDiffY_U2X = 2,   // difference.py:236                                mask X strict
  kDiffX_V2X = 3,   // difference.py:258                                mask X strict
  kDiffY_X2U = 4,   // difference.py:280  (q[j,i]-q[j-1,i])/dy         mask u
  kDiffX_X2V = 5,   // difference.py:301  (q[j,i]-q[j,i-1])/dx         mask v
  kDiffX_U2T = 6,   // difference.py:326                                mask h
  kDiffY_V2T = 7,   // difference.py:347                                mask h
  kDivergence = 8,  // difference.py:372 / _divergence_2d :62          mask h
  kDivNoflux = 9,   // divergence.py:138 (wall faces zeroed first)      mask h
  kCurl = 10,       // difference.py:401 / _curl_2d :47                 mask X strict
  kLaplacian = 11,  // difference.py:431                                mask h
  kGradPerpU = 12,  // difference.py:503-507                            mask u
  kGradPerpV = 13,  // difference.py:510-514                            mask v
  kT2X = 14,        // interpolation.py:158                             mask X strict
  kV2T = 15,        // interpolation.py:206                             mask h
  kNumOps = 16,
};

// A wavefront takes 64 columns x R rows: every load of its rows is in flight
// before the first result, and the rows share what they both read.  Fields of
// kManyCells and more (more than two rounds of wavefronts at a row each) take
// R = 2 in FP64 and 4 in FP32, smaller ones R = 1 (more wavefronts, shorter
// chains).  Masks are a template argument, so that their loads join the batch.
// Bound: bytes, beyond the 2.2 us of a launch.  us in a captured graph, a
// thread a point -> now:
//   curl, FP64 masked  1023 x 1535   9.0 -> 8.1   2000^2 19.7 -> 18.0
//   laplacian, FP32    1023 x 1535   4.2 -> 4.0   2000^2  9.7 ->  7.9
//   grad_perp (two launches before) FP64 masked 13.8 -> 10.0, 33.0 -> 23.2
//   diffusion, FP64 masked, kappa field 17.1 -> 10.1, 37.2 -> 23.7
// Rows tried at 2000^2: FP64 laplacian 14.6 with 1, 14.5 with 2, 15.2 with 4;
// FP32 9.7, 8.3, 7.9; at 500^2, FP64 masked, 2.8 with 1, 3.2 with 4.
template <typename T>
constexpr int kRows = sizeof(T) == 8 ? 2 : 4;
constexpr int64_t kManyCells = 1 << 19;

// Row and column of the stencil's centre: its own where the cell has one, else
// the nearest that has (the loads stay inside the array, the result is not
// used).
__device__ __forceinline__ int clamp_to(int x, int lo, int hi) { return min(max(x, lo), hi); }

template <typename T, int OP>
__device__ __forceinline__ T point_at(const T* __restrict__ a, const T* __restrict__ b, int64_t c,
                                      int j, int i, int ny, int nx, T idx, T idy) {
  T v = T(0);
  if constexpr (OP == kDiffX_T2U || OP == kDiffX_V2X) {
    v = (a[c + 1] - a[c]) * idx;
  } else if constexpr (OP == kDiffY_T2V || OP == kDiffY_U2X) {
    v = (a[c + nx] - a[c]) * idy;
  } else if constexpr (OP == kDiffY_X2U || OP == kDiffY_V2T) {
    v = (a[c] - a[c - nx]) * idy;
  } else if constexpr (OP == kDiffX_X2V || OP == kDiffX_U2T) {
    v = (a[c] - a[c - 1]) * idx;
  } else if constexpr (OP == kDivergence) {
    v = (a[c] - a[c - 1]) * idx + (b[c] - b[c - nx]) * idy;
  } else if constexpr (OP == kDivNoflux) {
    // u[:,0] = u[:,-2] = 0 and v[0,:] = v[-2,:] = 0 before the divergence.
    const T ue = (i == nx - 2) ? T(0) : a[c];
    const T uw = (i - 1 == 0) ? T(0) : a[c - 1];
    const T vn = (j == ny - 2) ? T(0) : b[c];
    const T vs = (j - 1 == 0) ? T(0) : b[c - nx];
    v = (ue - uw) * idx + (vn - vs) * idy;
  } else if constexpr (OP == kCurl) {
    v = (b[c + 1] - b[c]) * idx - (a[c + nx] - a[c]) * idy;
  } else if constexpr (OP == kLaplacian) {
    const T h0 = a[c];
    v = ((a[c + 1] - h0) - (h0 - a[c - 1])) * (idx * idx) +
        ((a[c + nx] - h0) - (h0 - a[c - nx])) * (idy * idy);
  } else if constexpr (OP == kGradPerpU) {
    v = -(a[c + nx] + a[c + nx + 1] - a[c - nx] - a[c - nx + 1]) * (T(0.25) * idy);
  } else if constexpr (OP == kGradPerpV) {
    v = (a[c + 1] + a[c + nx + 1] - a[c - 1] - a[c + nx - 1]) * (T(0.25) * idx);
  } else if constexpr (OP == kT2X) {
    v = T(0.25) * (a[c] + a[c + 1] + a[c + nx] + a[c + nx + 1]);
  } else if constexpr (OP == kV2T) {
    v = T(0.5) * (a[c] + a[c - nx]);
  }
  return v;
}

// INNER: all rows of the strip are interior (no row is clamped, so that rows
// share their loads).
template <typename T, int OP, int R, bool MASKED, bool INNER>
__device__ __forceinline__ void point_rows(const T* __restrict__ a, const T* __restrict__ b,
                                           T* __restrict__ out, const uint8_t* __restrict__ mask,
                                           int j0, int i, int ny, int nx, T idx, T idy) {
  const int ic = clamp_to(i, 1, nx - 2), il = min(i, nx - 1);
  T v[R];
  int m[R];
#pragma unroll
  for (int t = 0; t < R; ++t) {
    const int j = j0 + t, jc = INNER ? j : clamp_to(j, 1, ny - 2);
    if constexpr (MASKED) m[t] = (mask + (int64_t)(INNER ? j : min(j, ny - 1)) * nx)[il];
    v[t] = point_at<T, OP>(a, b, (int64_t)jc * nx + ic, jc, ic, ny, nx, idx, idy);
  }
#pragma unroll
  for (int t = 0; t < R; ++t) {
    const int j = j0 + t;
    if (i >= nx || (!INNER && j >= ny)) continue;
    T r = (INNER || (j >= 1 && j <= ny - 2)) && i >= 1 && i <= nx - 2 ? v[t] : T(0);
    if constexpr (MASKED) r = r * (T)(m[t] ? 1 : 0);
    out[(int64_t)j * nx + i] = r;
  }
}

template <typename T, int OP, int R, bool MASKED>
__global__ __launch_bounds__(256) void point_stencil_kernel(
    const T* __restrict__ a, const T* __restrict__ b, T* __restrict__ out,
    const uint8_t* __restrict__ mask, int ny, int nx, T idx, T idy) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  const int j0 = __builtin_amdgcn_readfirstlane((blockIdx.y * 4 + threadIdx.y) * R);
  if (j0 >= ny) return;
  if (j0 >= 1 && j0 + R <= ny - 1)
    point_rows<T, OP, R, MASKED, true>(a, b, out, mask, j0, i, ny, nx, idx, idy);
  else
    point_rows<T, OP, R, MASKED, false>(a, b, out, mask, j0, i, ny, nx, idx, idy);
}

// Both components of grad_perp in one pass over psi.
template <typename T, int R, bool MASKED>
__global__ __launch_bounds__(256) void grad_perp_kernel(const T* __restrict__ psi,
                                                        T* __restrict__ u, T* __restrict__ v,
                                                        const uint8_t* __restrict__ mu,
                                                        const uint8_t* __restrict__ mv, int ny,
                                                        int nx, T idx, T idy) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  const int j0 = __builtin_amdgcn_readfirstlane((blockIdx.y * 4 + threadIdx.y) * R);
  if (j0 >= ny) return;
  if (j0 >= 1 && j0 + R <= ny - 1) {
    point_rows<T, kGradPerpU, R, MASKED, true>(psi, nullptr, u, mu, j0, i, ny, nx, idx, idy);
    point_rows<T, kGradPerpV, R, MASKED, true>(psi, nullptr, v, mv, j0, i, ny, nx, idx, idy);
  } else {
    point_rows<T, kGradPerpU, R, MASKED, false>(psi, nullptr, u, mu, j0, i, ny, nx, idx, idy);
    point_rows<T, kGradPerpV, R, MASKED, false>(psi, nullptr, v, mv, j0, i, ny, nx, idx, idy);
  }
}

static inline bool many_rows(int ny, int nx) { return (int64_t)ny * nx >= kManyCells; }
static inline dim3 rows_grid(int ny, int nx, int rows) {
  return dim3(cdiv(nx, 64), cdiv(ny, 4 * rows));
}

template <typename T>
using PointKernel = void (*)(const T*, const T*, T*, const uint8_t*, int, int, T, T);

template <typename T, int R, bool MASKED, int... OPS>
struct PointTable {
  static constexpr PointKernel<T> table[] = {&point_stencil_kernel<T, OPS, R, MASKED>...};
};

template <typename T>
int point_stencil(int op, const T* a, const T* b, T* out, int ny, int nx, double dx,
                  double dy, const uint8_t* mask, hipStream_t s) {
  FVX_CHECK_ARG(op >= 0 && op < kNumOps, "unknown stencil op %d", op);
  FVX_CHECK_ARG(a && out, "null field pointer");
  FVX_CHECK_ARG(ny >= 3 && nx >= 3, "array too small (%d x %d); need >= 3 x 3", ny, nx);
  FVX_CHECK_ARG(dx > 0 && dy > 0, "grid spacing must be positive");
  const bool two = (op == kDivergence || op == kDivNoflux || op == kCurl);
  FVX_CHECK_ARG(!two || b, "operator needs a second field");
  const bool many = many_rows(ny, nx);
#define FVX_OPS 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15
  const PointKernel<T> k = many ? (mask ? PointTable<T, kRows<T>, true, FVX_OPS>::table[op]
                                        : PointTable<T, kRows<T>, false, FVX_OPS>::table[op])
                                : (mask ? PointTable<T, 1, true, FVX_OPS>::table[op]
                                        : PointTable<T, 1, false, FVX_OPS>::table[op]);
#undef FVX_OPS
  hipLaunchKernelGGL(k, rows_grid(ny, nx, many ? kRows<T> : 1), dim3(64, 4), 0, s, a, b, out, mask, ny,
                     nx, (T)(1.0 / dx), (T)(1.0 / dy));
  FVX_LAUNCH_CHECK();
  return kOk;
}

template <typename T>
int grad_perp(const T* psi, T* u, T* v, int ny, int nx, double dx, double dy, const uint8_t* mu,
              const uint8_t* mv, hipStream_t s) {
  FVX_CHECK_ARG(psi && u && v, "null field pointer");
  FVX_CHECK_ARG(ny >= 3 && nx >= 3, "array too small (%d x %d); need >= 3 x 3", ny, nx);
  FVX_CHECK_ARG(dx > 0 && dy > 0, "grid spacing must be positive");
  FVX_CHECK_ARG((mu == nullptr) == (mv == nullptr), "mask_u and mask_v go together");
  const bool many = many_rows(ny, nx);
  const dim3 g = rows_grid(ny, nx, many ? kRows<T> : 1), b(64, 4);
  const T ix = (T)(1.0 / dx), iy = (T)(1.0 / dy);
#define FVX_GP(R, M) \
  hipLaunchKernelGGL((grad_perp_kernel<T, R, M>), g, b, 0, s, psi, u, v, mu, mv, ny, nx, ix, iy)
  if (many && mu) FVX_GP(kRows<T>, true);
  else if (many) FVX_GP(kRows<T>, false);
  else if (mu) FVX_GP(1, true);
  else FVX_GP(1, false);
#undef FVX_GP
  FVX_LAUNCH_CHECK();
  return kOk;
}

// ---------------------------------------------------------------------------
// Diffusion2D (diffusion.py:120-176): face fluxes exist only strictly between
// interior cells (no-flux walls); masked fluxes; tendency x mask.h.
// ---------------------------------------------------------------------------

template <typename T>
__device__ __forceinline__ T kappa_at(const T* kap, T k0, int64_t c) {
  return kap ? kap[c] : k0;
}

template <typename T>
__device__ __forceinline__ T flux_x_at(const T* h, const T* kap, T k0, const uint8_t* mu,
                                       int j, int i, int ny, int nx, T idx) {
  // flux_x[j, i+1/2] for i = 1..nx-3, rows 1..ny-2 (diffusion.py:151-155)
  if (j < 1 || j > ny - 2 || i < 1 || i > nx - 3) return T(0);
  const int64_t c = (int64_t)j * nx + i;
  T f = kappa_at(kap, k0, c) * (h[c + 1] - h[c]) * idx;
  if (mu) f = f * (T)(mu[c] ? 1 : 0);
  return f;
}

template <typename T>
__device__ __forceinline__ T flux_y_at(const T* h, const T* kap, T k0, const uint8_t* mv,
                                       int j, int i, int ny, int nx, T idy) {
  // flux_y[j+1/2, i] for j = 1..ny-3, cols 1..nx-2 (diffusion.py:159-165)
  if (j < 1 || j > ny - 3 || i < 1 || i > nx - 2) return T(0);
  const int64_t c = (int64_t)j * nx + i;
  T f = kappa_at(kap, k0, c) * (h[c + nx] - h[c]) * idy;
  if (mv) f = f * (T)(mv[c] ? 1 : 0);
  return f;
}

// FULL: all three masks are there (else each may be null).
template <typename T, int R, bool FULL, bool INNER>
__device__ __forceinline__ void diffusion_rows(const T* __restrict__ h, const T* __restrict__ kap,
                                               T k0, T* __restrict__ out,
                                               const uint8_t* __restrict__ mh,
                                               const uint8_t* __restrict__ mu,
                                               const uint8_t* __restrict__ mv, int j0, int i,
                                               int ny, int nx, T idx, T idy) {
  // rows j0 - 1 .. j0 + R of h; fluxes through the north faces of rows
  // j0 - 1 .. and through the west and east faces of rows j0 ..
  const int ic = clamp_to(i, 1, nx - 2), il = min(i, nx - 1);
  auto row = [&](int j) -> int64_t { return (int64_t)(INNER ? j : clamp_to(j, 0, ny - 1)) * nx; };
  T hc[R + 2], he[R], hw[R], kc[R + 1], kw[R];
  int nv[R + 1], ne[R], nw[R], nh[R];
#pragma unroll
  for (int t = 0; t < R + 2; ++t) hc[t] = (h + row(j0 - 1 + t))[ic];
#pragma unroll
  for (int t = 0; t < R + 1; ++t) {
    kc[t] = kap ? (kap + row(j0 - 1 + t))[ic] : k0;
    nv[t] = FULL || mv ? (mv + row(j0 - 1 + t))[ic] : 1;
  }
#pragma unroll
  for (int t = 0; t < R; ++t) {
    he[t] = (h + row(j0 + t))[ic + 1];
    hw[t] = (h + row(j0 + t))[ic - 1];
    kw[t] = kap ? (kap + row(j0 + t))[ic - 1] : k0;
    ne[t] = FULL || mu ? (mu + row(j0 + t))[ic] : 1;
    nw[t] = FULL || mu ? (mu + row(j0 + t))[ic - 1] : 1;
    nh[t] = FULL || mh ? (mh + row(j0 + t))[il] : 1;
  }
  T fn[R + 1];
#pragma unroll
  for (int t = 0; t < R + 1; ++t) {
    const int j = j0 - 1 + t;
    T f = kc[t] * (hc[t + 1] - hc[t]) * idy;
    if (FULL || mv) f = f * (T)(nv[t] ? 1 : 0);
    fn[t] = j >= 1 && j <= ny - 3 ? f : T(0);
  }
#pragma unroll
  for (int t = 0; t < R; ++t) {
    const int j = j0 + t;
    if (i >= nx || (!INNER && j >= ny)) continue;
    T fe = kc[t + 1] * (he[t] - hc[t + 1]) * idx, fw = kw[t] * (hc[t + 1] - hw[t]) * idx;
    if (FULL || mu) {
      fe = fe * (T)(ne[t] ? 1 : 0);
      fw = fw * (T)(nw[t] ? 1 : 0);
    }
    fe = i <= nx - 3 ? fe : T(0);
    fw = i >= 2 ? fw : T(0);
    T v = (fe - fw) * idx + (fn[t + 1] - fn[t]) * idy;
    if (!((INNER || (j >= 1 && j <= ny - 2)) && i >= 1 && i <= nx - 2)) v = T(0);
    if (FULL || mh) v = v * (T)(nh[t] ? 1 : 0);
    out[(int64_t)j * nx + i] = v;
  }
}

template <typename T, int R, bool FULL>
__global__ __launch_bounds__(256) void diffusion_kernel(
    const T* __restrict__ h, const T* __restrict__ kap, T k0, T* __restrict__ out,
    const uint8_t* __restrict__ mh, const uint8_t* __restrict__ mu,
    const uint8_t* __restrict__ mv, int ny, int nx, T idx, T idy) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  const int j0 = __builtin_amdgcn_readfirstlane((blockIdx.y * 4 + threadIdx.y) * R);
  if (j0 >= ny) return;
  if (j0 >= 1 && j0 + R <= ny - 1)
    diffusion_rows<T, R, FULL, true>(h, kap, k0, out, mh, mu, mv, j0, i, ny, nx, idx, idy);
  else
    diffusion_rows<T, R, FULL, false>(h, kap, k0, out, mh, mu, mv, j0, i, ny, nx, idx, idy);
}

template <typename T>
__global__ __launch_bounds__(256) void diffusion_fluxes_kernel(
    const T* __restrict__ h, const T* __restrict__ kap, T k0, T* __restrict__ fx,
    T* __restrict__ fy, const uint8_t* __restrict__ mu, const uint8_t* __restrict__ mv,
    int ny, int nx, T idx, T idy) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  const int j = blockIdx.y * 4 + threadIdx.y;
  if (i >= nx || j >= ny) return;
  const int64_t c = (int64_t)j * nx + i;
  fx[c] = flux_x_at(h, kap, k0, mu, j, i, ny, nx, idx);
  fy[c] = flux_y_at(h, kap, k0, mv, j, i, ny, nx, idy);
}

template <typename T>
int diffusion(const T* h, const T* kap, double k0, T* out, int ny, int nx, double dx,
              double dy, const uint8_t* mh, const uint8_t* mu, const uint8_t* mv,
              hipStream_t s) {
  FVX_CHECK_ARG(h && out, "null field pointer");
  FVX_CHECK_ARG(ny >= 3 && nx >= 3, "array too small (%d x %d)", ny, nx);
  FVX_CHECK_ARG(dx > 0 && dy > 0, "grid spacing must be positive");
  const bool many = many_rows(ny, nx), full = mh && mu && mv;
  const dim3 g = rows_grid(ny, nx, many ? kRows<T> : 1), b(64, 4);
  const T ix = (T)(1.0 / dx), iy = (T)(1.0 / dy);
#define FVX_DIFF(R, F)                                                                          \
  hipLaunchKernelGGL((diffusion_kernel<T, R, F>), g, b, 0, s, h, kap, (T)k0, out, mh, mu, mv, \
                     ny, nx, ix, iy)
  if (many && full) FVX_DIFF(kRows<T>, true);
  else if (many) FVX_DIFF(kRows<T>, false);
  else if (full) FVX_DIFF(1, true);
  else FVX_DIFF(1, false);
#undef FVX_DIFF
  FVX_LAUNCH_CHECK();
  return kOk;
}

template <typename T>
int diffusion_fluxes(const T* h, const T* kap, double k0, T* fx, T* fy, int ny, int nx,
                     double dx, double dy, const uint8_t* mu, const uint8_t* mv,
                     hipStream_t s) {
  FVX_CHECK_ARG(h && fx && fy, "null field pointer");
  FVX_CHECK_ARG(ny >= 3 && nx >= 3, "array too small (%d x %d)", ny, nx);
  FVX_CHECK_ARG(dx > 0 && dy > 0, "grid spacing must be positive");
  dim3 blk(64, 4), grd(cdiv(nx, 64), cdiv(ny, 4));
  hipLaunchKernelGGL(diffusion_fluxes_kernel<T>, grd, blk, 0, s, h, kap, (T)k0, fx, fy, mu,
                     mv, ny, nx, (T)(1.0 / dx), (T)(1.0 / dy));
  FVX_LAUNCH_CHECK();
  return kOk;
}

// ---------------------------------------------------------------------------
// Fused BiharmonicDiffusion2D (diffusion.py:543-574): -kappa * D(D(h)) with the
// unmasked no-flux Laplacian D applied twice; the intermediate never touches
// HBM.  Traffic: read h, write out (2 x sizeof T
// per cell, + 1 byte when masked).
// ---------------------------------------------------------------------------

// One wavefront per 60 columns x R rows: a lane holds column i of h on
// rows j0 - 2 .. j0 + R + 1, the inner Laplacian stays in registers, the
// east and west values are lane moves: one pass, no LDS and no barriers (an
// LDS tile with integer divisions a cell: us, FP64 1023 x 1535 11.0 -> 6.9, 2000^2
// 25.5 -> 12.4; FP32 9.9 -> 4.8, 21.4 -> 7.8).  8 rows, 2 below kManyCells (500^2
// FP64 4.0 -> 3.2).  The fluxes between
// two cells exist only when both are interior.
constexpr int kBhCols = 60;

template <typename T, int R, bool MASKED>
__global__ __launch_bounds__(256) void biharmonic_kernel(
    const T* __restrict__ h, T* __restrict__ out, const uint8_t* __restrict__ mh, int ny,
    int nx, T idx, T idy, T kappa, int tiles_x, int ntiles) {
  const int lane = threadIdx.x & 63;
  const int t = __builtin_amdgcn_readfirstlane(xcd_swizzle(blockIdx.x, gridDim.x) * 4 +
                                               (threadIdx.x >> 6));
  if (t >= ntiles) return;  // whole wavefront
  const int ty = t / tiles_x, j0 = ty * R, i = (t - ty * tiles_x) * kBhCols - 2 + lane;
  const unsigned ic = (unsigned)min(max(i, 0), nx - 1);
  T hr[R + 4];
  int m[MASKED ? R : 1];
#pragma unroll
  for (int r = 0; r < R + 4; ++r)
    hr[r] = (h + (int64_t)min(max(j0 - 2 + r, 0), ny - 1) * nx)[ic];
  if constexpr (MASKED) {
#pragma unroll
    for (int r = 0; r < R; ++r) m[r] = (mh + (int64_t)min(j0 + r, ny - 1) * nx)[ic];
  }
  const bool in = i >= 1 && i <= nx - 2, east = in && i <= nx - 3;
  // D at row j of the field whose rows south, centre and north are s, c, n
  auto lap = [&](T s, T c, T n, int j) -> T {
    const T de = (dpp_move<0x130>(c) - c) * idx;  // (moved with all lanes active)
    const T fe = east ? de : T(0), fw = dpp_move<0x138>(fe);
    const T fn = j <= ny - 3 ? (n - c) * idy : T(0), fs = j >= 2 ? (c - s) * idy : T(0);
    return in && j >= 1 && j <= ny - 2 ? (fe - fw) * idx + (fn - fs) * idy : T(0);
  };
  T l[R + 2];
#pragma unroll
  for (int r = 0; r < R + 2; ++r) l[r] = lap(hr[r], hr[r + 1], hr[r + 2], j0 - 1 + r);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int j = j0 + r;
    T v = -kappa * lap(l[r], l[r + 1], l[r + 2], j);
    if constexpr (MASKED) v = v * (T)(m[r] ? 1 : 0);
    if (j < ny && lane >= 2 && lane < 62 && i < nx) (out + (int64_t)j * nx)[i] = v;
  }
}

template <typename T>
int biharmonic(const T* h, T* out, int ny, int nx, double dx, double dy, double kappa,
               const uint8_t* mh, hipStream_t s) {
  FVX_CHECK_ARG(h && out, "null field pointer");
  FVX_CHECK_ARG(ny >= 3 && nx >= 3, "array too small (%d x %d)", ny, nx);
  FVX_CHECK_ARG(dx > 0 && dy > 0, "grid spacing must be positive");
  const bool many = many_rows(ny, nx);
  const int tx = cdiv(nx, kBhCols), nt = tx * cdiv(ny, many ? 8 : 2);
  const dim3 grd(cdiv(nt, 4)), blk(256);
  const T ix = (T)(1.0 / dx), iy = (T)(1.0 / dy);
#define FVX_BIH(R, M)                                                                            \
  hipLaunchKernelGGL((biharmonic_kernel<T, R, M>), grd, blk, 0, s, h, out, mh, ny, nx, ix, iy, \
                     (T)kappa, tx, nt)
  if (many && mh) FVX_BIH(8, true);
  else if (many) FVX_BIH(8, false);
  else if (mh) FVX_BIH(2, true);
  else FVX_BIH(2, false);
#undef FVX_BIH
  FVX_LAUNCH_CHECK();
  return kOk;
}

// ---------------------------------------------------------------------------
// Arakawa (1966) Jacobian (jacobian.py:22-131): interior-only output
// (batch, ny-2, nx-2); inputs (batch, ny, nx).  The three forms are summed in
// the reference's order and divided by 12 dx dy.
// ---------------------------------------------------------------------------

// One wavefront per 62 output columns x R output rows, a lane a column of f and
// g: 2 (R + 2) / R loads a point instead of 16; the columns beside it are lane
// moves.  4 rows (2 below kManyCells).  us, a thread a point -> now: FP64 1023 x
// 1535 11.5 -> 7.4, 2000^2 25.9 -> 15.7, 500^2 3.5 -> 3.2; FP32 6.5 -> 5.0, 12.8 ->
// 9.3, 2.6 -> 2.8.
constexpr int kJacCols = 62;

template <typename T, int R>
__global__ __launch_bounds__(256) void arakawa_kernel(const T* __restrict__ f,
                                                      const T* __restrict__ g,
                                                      T* __restrict__ out, int ny, int nx,
                                                      T scale, int tiles_x, int ntiles) {
  const int lane = threadIdx.x & 63;
  const int t = __builtin_amdgcn_readfirstlane(xcd_swizzle(blockIdx.x, gridDim.x) * 4 +
                                               (threadIdx.x >> 6));
  if (t >= ntiles) return;  // whole wavefront
  const int64_t base = (int64_t)blockIdx.y * ny * nx;
  const int ty = t / tiles_x, j0 = ty * R;                // input rows j0 .. j0 + R + 1
  const int i = (t - ty * tiles_x) * kJacCols + lane;     // input column
  const unsigned ic = (unsigned)min(i, nx - 1);
  T fc[R + 2], gc[R + 2];
#pragma unroll
  for (int r = 0; r < R + 2; ++r) {
    const int64_t o = base + (int64_t)min(j0 + r, ny - 1) * nx;
    fc[r] = (f + o)[ic];
    gc[r] = (g + o)[ic];
  }
  T fe[R + 2], fw[R + 2], ge[R + 2], gw[R + 2];
#pragma unroll
  for (int r = 0; r < R + 2; ++r) {
    fe[r] = dpp_move<0x130>(fc[r]);
    fw[r] = dpp_move<0x138>(fc[r]);
    ge[r] = dpp_move<0x130>(gc[r]);
    gw[r] = dpp_move<0x138>(gc[r]);
  }
  const bool col = lane >= 1 && lane <= 62 && i <= nx - 2;
  out += (int64_t)blockIdx.y * (ny - 2) * (nx - 2);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const T fE = fe[r + 1], fW = fw[r + 1], fN = fc[r + 2], fS = fc[r];
    const T fNE = fe[r + 2], fNW = fw[r + 2], fSE = fe[r], fSW = fw[r];
    const T gE = ge[r + 1], gW = gw[r + 1], gN = gc[r + 2], gS = gc[r];
    const T gNE = ge[r + 2], gNW = gw[r + 2], gSE = ge[r], gSW = gw[r];
    const T jpp = (fE - fW) * (gN - gS) - (fN - fS) * (gE - gW);
    const T jpx = fE * (gNE - gSE) - fW * (gNW - gSW) - fN * (gNE - gNW) + fS * (gSE - gSW);
    const T jxp = gN * (fNE - fNW) - gS * (fSE - fSW) - gE * (fNE - fSE) + gW * (fNW - fSW);
    if (col && j0 + r < ny - 2)
      (out + (int64_t)(j0 + r) * (nx - 2))[i - 1] = ((jpp + jpx) + jxp) / scale;
  }
}

template <typename T>
int arakawa(const T* f, const T* g, T* out, int batch, int ny, int nx, double dx, double dy,
            hipStream_t s) {
  FVX_CHECK_ARG(f && g && out, "null field pointer");
  FVX_CHECK_ARG(batch >= 1 && batch <= 65535, "batch must be in [1, 65535], got %d", batch);
  FVX_CHECK_ARG(ny >= 3 && nx >= 3, "array too small (%d x %d)", ny, nx);
  const bool many = many_rows(ny, nx);
  const int tx = cdiv(nx - 2, kJacCols), nt = tx * cdiv(ny - 2, many ? 4 : 2);
  const dim3 grd(cdiv(nt, 4), batch), blk(256);
  const T scale = (T)(12.0 * dx * dy);
  if (many)
    hipLaunchKernelGGL((arakawa_kernel<T, 4>), grd, blk, 0, s, f, g, out, ny, nx, scale, tx, nt);
  else
    hipLaunchKernelGGL((arakawa_kernel<T, 2>), grd, blk, 0, s, f, g, out, ny, nx, scale, tx, nt);
  FVX_LAUNCH_CHECK();
  return kOk;
}

// ---------------------------------------------------------------------------
// masked_laplacian (iterative.py:144-191): Dirichlet outside the mask with a
// periodic roll at the array edge; the mask is a field of the same dtype.
// ---------------------------------------------------------------------------

template <typename T>
__global__ __launch_bounds__(256) void masked_laplacian_kernel(
    const T* __restrict__ psi, const T* __restrict__ mask, T* __restrict__ out, int ny,
    int nx, T idx2, T idy2, T lam) {
  const int i = blockIdx.x * 64 + threadIdx.x;
  const int j = blockIdx.y * 4 + threadIdx.y;
  if (i >= nx || j >= ny) return;
  const int ie = (i + 1 == nx) ? 0 : i + 1, iw = (i == 0) ? nx - 1 : i - 1;
  const int jn = (j + 1 == ny) ? 0 : j + 1, js = (j == 0) ? ny - 1 : j - 1;
  auto pm = [&](int jj, int ii) {
    const int64_t k = (int64_t)jj * nx + ii;
    return psi[k] * mask[k];
  };
  const T p = pm(j, i);
  const T lap = (pm(j, iw) + pm(j, ie) - T(2) * p) * idx2 + (pm(js, i) + pm(jn, i) - T(2) * p) * idy2;
  out[(int64_t)j * nx + i] = (lap - lam * p) * mask[(int64_t)j * nx + i];
}

template <typename T>
int masked_laplacian(const T* psi, const T* mask, T* out, int ny, int nx, double dx,
                     double dy, double lam, hipStream_t s) {
  FVX_CHECK_ARG(psi && mask && out, "null field pointer");
  FVX_CHECK_ARG(ny >= 1 && nx >= 1, "empty array");
  dim3 blk(64, 4), grd(cdiv(nx, 64), cdiv(ny, 4));
  hipLaunchKernelGGL(masked_laplacian_kernel<T>, grd, blk, 0, s, psi, mask, out, ny, nx,
                     (T)(1.0 / (dx * dx)), (T)(1.0 / (dy * dy)), (T)lam);
  FVX_LAUNCH_CHECK();
  return kOk;
}

// ---------------------------------------------------------------------------
// Periodic ghost fill of width ng (boundary.py:52-78), in place, in one
// launch: every ghost cell copies the interior cell its row and column wrap
// to (the reference fills rows, then columns, so a corner takes the
// diagonally opposite interior value: the same cell).  Reads touch interior
// cells only and writes ghost cells only, so the threads do not race.
// ---------------------------------------------------------------------------

__device__ __forceinline__ int periodic_wrap(int x, int n, int ng) {
  return x < ng ? x + n - 2 * ng : (x >= n - ng ? x - n + 2 * ng : x);
}

template <typename T>
__global__ __launch_bounds__(256) void periodic_fill_kernel(T* f, int ny, int nx, int ng) {
  // cells 0 .. 2 ng nx - 1: the ghost rows (full width); then the ghost
  // columns of the interior rows, 2 ng per row
  const int64_t nrow = 2LL * ng * nx, ncol = 2LL * ng * (ny - 2 * ng);
  const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int j, i;
  if (k < nrow) {
    const int g = (int)(k / nx);
    i = (int)(k - (int64_t)g * nx);
    j = g < ng ? g : ny - 2 * ng + g;
  } else if (k < nrow + ncol) {
    const int64_t q = k - nrow;
    const int r = (int)(q / (2 * ng)), g = (int)(q - (int64_t)r * 2 * ng);
    j = ng + r;
    i = g < ng ? g : nx - 2 * ng + g;
  } else {
    return;
  }
  f[(int64_t)j * nx + i] = f[(int64_t)periodic_wrap(j, ny, ng) * nx + periodic_wrap(i, nx, ng)];
}

template <typename T>
int enforce_periodic(T* f, int ny, int nx, int ng, hipStream_t s) {
  FVX_CHECK_ARG(f, "null field pointer");
  FVX_CHECK_ARG(ng >= 1 && ny >= 3 * ng && nx >= 3 * ng,
                "ghost width %d too large for %d x %d", ng, ny, nx);
  const int64_t cells = 2LL * ng * nx + 2LL * ng * (ny - 2 * ng);
  hipLaunchKernelGGL(periodic_fill_kernel<T>, dim3((unsigned)((cells + 255) / 256)), dim3(256), 0,
                     s, f, ny, nx, ng);
  FVX_LAUNCH_CHECK();
  return kOk;
}

// ---------------------------------------------------------------------------
// The double-gyre example's tendency (scripts/qg_1p5_layer.py:454-478) and
// velocities (:115-145) in one pass, with the fields' composition of the
// operators above: X = T_to_X(psi), u = -diff_y_X_to_U(X), v = diff_x_X_to_V(X),
//   rhs = advection(q; upwind1) - beta V_to_T(v) + wind
//         - drag laplacian(psi) + viscosity laplacian(q)
// (every operator's ghost ring zero, the advection's two cells wide; wind on
// every cell).  One thread a cell: the velocities around the cell take the nine
// psi values around it, so nothing is exchanged.  Why: as the eight operator
// calls it was one short launch each, all bound by the host's time per call
// (64^2 step: 382 us so, 158 with this kernel and the inversion from field to
// field).  q null: velocities only.
// ---------------------------------------------------------------------------
template <typename T>
struct GyreArgs {
  const T *q, *psi, *wind;
  T *rhs, *u, *v;
  int ny, nx;
  T idx, idy, beta, drag, visc;
};

template <typename T>
__global__ __launch_bounds__(256) void gyre_kernel(GyreArgs<T> g) {
  const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
  const int ny = g.ny, nx = g.nx;
  if (i >= nx || j >= ny) return;
  const int64_t c = (int64_t)j * nx + i;
  const bool in = j >= 1 && j <= ny - 2 && i >= 1 && i <= nx - 2;
  T u0 = T(0), v0 = T(0), rhs = T(0);
  if (in) {
    T p[3][3];
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
      for (int a = 0; a < 3; ++a) p[b][a] = g.psi[c + (int64_t)(b - 1) * nx + (a - 1)];
    // X[b][a] at (j - 1 + b, i - 1 + a), zero on the ring
    T X[2][2];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int a = 0; a < 2; ++a)
        X[b][a] = j - 1 + b >= 1 && i - 1 + a >= 1
                      ? T(0.25) * (p[b][a] + p[b][a + 1] + p[b + 1][a] + p[b + 1][a + 1])
                      : T(0);
    u0 = -((X[1][1] - X[0][1]) * g.idy);
    v0 = (X[1][1] - X[1][0]) * g.idx;
    if (g.q) {
      const T uw = -((X[1][0] - X[0][0]) * g.idy), vs = (X[0][1] - X[0][0]) * g.idx;
      const T q0 = g.q[c], qe = g.q[c + 1], qw = g.q[c - 1], qn = g.q[c + nx], qs = g.q[c - nx];
      T adv = T(0);
      if (j >= 2 && j <= ny - 3 && i >= 2 && i <= nx - 3) {
        const T fe = (u0 >= T(0) ? q0 : qe) * u0, fw = (uw >= T(0) ? qw : q0) * uw;
        const T fn = (v0 >= T(0) ? q0 : qn) * v0, fs = (vs >= T(0) ? qs : q0) * vs;
        adv = -((fe - fw) * g.idx + (fn - fs) * g.idy);
      }
      const T zeta = ((p[1][2] - p[1][1]) - (p[1][1] - p[1][0])) * (g.idx * g.idx) +
                     ((p[2][1] - p[1][1]) - (p[1][1] - p[0][1])) * (g.idy * g.idy);
      const T lq = ((qe - q0) - (q0 - qw)) * (g.idx * g.idx) +
                   ((qn - q0) - (q0 - qs)) * (g.idy * g.idy);
      rhs = (adv - g.beta * (T(0.5) * (v0 + vs))) - g.drag * zeta + g.visc * lq;
    }
  }
  g.u[c] = u0;
  g.v[c] = v0;
  if (g.q) g.rhs[c] = rhs + g.wind[c];
}

template <typename T>
static int gyre(const T* q, const T* psi, const T* wind, T* rhs, T* u, T* v, int ny, int nx,
                double dx, double dy, double beta, double drag, double visc, hipStream_t s) {
  FVX_CHECK_ARG(psi && u && v, "null field pointer");
  FVX_CHECK_ARG(!q || (wind && rhs), "the tendency needs the wind field and an output");
  FVX_CHECK_ARG(ny >= 3 && nx >= 3, "array too small (%d x %d); need >= 3 x 3", ny, nx);
  FVX_CHECK_ARG(!q || (ny >= 5 && nx >= 5), "advection needs at least 5 x 5 (%d x %d)", ny, nx);
  FVX_CHECK_ARG(dx > 0 && dy > 0, "grid spacing must be positive");
  const GyreArgs<T> g{q,  psi, wind, rhs, u, v, ny, nx, (T)(1.0 / dx), (T)(1.0 / dy), (T)beta,
                      (T)drag, (T)visc};
  hipLaunchKernelGGL(gyre_kernel<T>, dim3(cdiv(nx, 64), cdiv(ny, 4)), dim3(64, 4), 0, s, g);
  FVX_LAUNCH_CHECK();
  return kOk;
}

}  // namespace fvx

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
extern "C" {

#define FVX_DT(SUF, T)                                                                      \
  int fvx_stencil2d_##SUF(int op, const T* a, const T* b, T* out, int ny, int nx,           \
                          double dx, double dy, const uint8_t* mask, void* stream) {        \
    return fvx::point_stencil<T>(op, a, b, out, ny, nx, dx, dy, mask, (hipStream_t)stream); \
  }                                                                                         \
  int fvx_grad_perp_##SUF(const T* psi, T* u, T* v, int ny, int nx, double dx, double dy,   \
                          const uint8_t* mu, const uint8_t* mv, void* stream) {             \
    return fvx::grad_perp<T>(psi, u, v, ny, nx, dx, dy, mu, mv, (hipStream_t)stream);       \
  }                                                                                         \
  int fvx_diffusion2d_##SUF(const T* h, const T* kappa, double kappa0, T* out, int ny,      \
                            int nx, double dx, double dy, const uint8_t* mh,                \
                            const uint8_t* mu, const uint8_t* mv, void* stream) {           \
    return fvx::diffusion<T>(h, kappa, kappa0, out, ny, nx, dx, dy, mh, mu, mv,             \
                             (hipStream_t)stream);                                          \
  }                                                                                         \
  int fvx_diffusion2d_fluxes_##SUF(const T* h, const T* kappa, double kappa0, T* fx, T* fy, \
                                   int ny, int nx, double dx, double dy, const uint8_t* mu, \
                                   const uint8_t* mv, void* stream) {                       \
    return fvx::diffusion_fluxes<T>(h, kappa, kappa0, fx, fy, ny, nx, dx, dy, mu, mv,       \
                                    (hipStream_t)stream);                                   \
  }                                                                                         \
  int fvx_biharmonic2d_##SUF(const T* h, T* out, int ny, int nx, double dx, double dy,      \
                             double kappa, const uint8_t* mh, void* stream) {               \
    return fvx::biharmonic<T>(h, out, ny, nx, dx, dy, kappa, mh, (hipStream_t)stream);      \
  }                                                                                         \
  int fvx_arakawa_jacobian_##SUF(const T* f, const T* g, T* out, int batch, int ny, int nx, \
                                 double dx, double dy, void* stream) {                      \
    return fvx::arakawa<T>(f, g, out, batch, ny, nx, dx, dy, (hipStream_t)stream);          \
  }                                                                                         \
  int fvx_masked_laplacian_##SUF(const T* psi, const T* mask, T* out, int ny, int nx,       \
                                 double dx, double dy, double lambda_, void* stream) {      \
    return fvx::masked_laplacian<T>(psi, mask, out, ny, nx, dx, dy, lambda_,                \
                                    (hipStream_t)stream);                                   \
  }                                                                                         \
  int fvx_enforce_periodic_##SUF(T* field, int ny, int nx, int ng, void* stream) {          \
    return fvx::enforce_periodic<T>(field, ny, nx, ng, (hipStream_t)stream);                \
  }                                                                                         \
  int fvx_gyre_tendency_##SUF(const T* q, const T* psi, const T* wind, T* rhs, T* u, T* v,  \
                              int ny, int nx, double dx, double dy, double beta,            \
                              double drag, double viscosity, void* stream) {                \
    return fvx::gyre<T>(q, psi, wind, rhs, u, v, ny, nx, dx, dy, beta, drag, viscosity,     \
                        (hipStream_t)stream);                                               \
  }

FVX_DT(f32, float)
FVX_DT(f64, double)
#undef FVX_DT
}
