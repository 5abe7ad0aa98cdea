// Vector-invariant momentum advection (MomentumAdvection2D.__call__,
// diffusion/momentum.py:37-248): du = +(zeta v)_u - dK/dx at U points,
// dv = -(zeta u)_v - dK/dy at V points, written on [2:-2, 2:-2] (zero
// elsewhere), with zeta = curl(u, v) at X points, K = (u_T^2 + v_T^2) / 2 at
// T points and the vorticity flux in Sadourny's energy or enstrophy form or
// the Arakawa-Lamb blend (1/3 energy + 2/3 enstrophy).  With a mask every
// intermediate is multiplied by the mask of its stagger, as the reference's
// masked Difference2D / Interpolation2D do, and the result by mask.u / mask.v.
//
// A wavefront takes 62 columns x R rows: a lane holds column i of u, v and the
// masks on rows j0 - 1 .. j0 + R; what a point needs of the columns beside it
// (u, v, the vorticity, K, the averaged u) are lane moves.  No intermediate
// reaches HBM; traffic per cell is read u, v, write du, dv (+ 4 mask bytes).
// (A thread a point loaded 14 values and 8 mask bytes each.)  Bound: bytes.  us in
// a captured graph, Arakawa-Lamb, then -> now: masked FP64 1023 x 1535 13.5 ->
// 10.8, 2000^2 32.9 -> 22.7; masked FP32 9.7 -> 7.4, 20.8 -> 14.5.

#include "fvx_common.hpp"

namespace fvx {

enum MomentumScheme : int { kEnergy = 0, kEnstrophy = 1, kArakawaLamb = 2 };

constexpr int kMomCols = 62;

template <typename T, int SCHEME, bool MASKED, int R>
__global__ __launch_bounds__(256) void momentum_kernel(
    const T* __restrict__ u, const T* __restrict__ v, T* __restrict__ du, T* __restrict__ dv,
    const uint8_t* __restrict__ mh, const uint8_t* __restrict__ mu,
    const uint8_t* __restrict__ mv, const uint8_t* __restrict__ mq, int ny, int nx, T idx,
    T idy, int tiles_x, int ntiles) {
  constexpr bool ENS = SCHEME != kEnergy;
  const int lane = threadIdx.x & 63;
  const int t = __builtin_amdgcn_readfirstlane(xcd_swizzle(blockIdx.x, gridDim.x) * 4 +
                                               (threadIdx.x >> 6));
  if (t >= ntiles) return;  // whole wavefront
  const int ty = t / tiles_x, j0 = ty * R, i = (t - ty * tiles_x) * kMomCols - 1 + lane;
  const unsigned ic = (unsigned)min(max(i, 0), nx - 1);
  auto row = [&](int j) -> int64_t { return (int64_t)min(max(j, 0), ny - 1) * nx; };
  auto east = [](T x) -> T { return dpp_move<0x130>(x); };
  auto west = [](T x) -> T { return dpp_move<0x138>(x); };
  // Index r: row j0 - 1 + r of u, v, mq; row j0 + r of mh, mu, mv.
  T uc[R + 2], vc[R + 2];
  int bq[MASKED ? R + 1 : 1], bh[MASKED ? R + 1 : 1], bu[MASKED ? R : 1], bv[MASKED ? R : 1];
#pragma unroll
  for (int r = 0; r < R + 2; ++r) {
    uc[r] = (u + row(j0 - 1 + r))[ic];
    vc[r] = (v + row(j0 - 1 + r))[ic];
  }
  if constexpr (MASKED) {
#pragma unroll
    for (int r = 0; r < R + 1; ++r) {
      bq[r] = (mq + row(j0 - 1 + r))[ic];
      bh[r] = (mh + row(j0 + r))[ic];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      bu[r] = (mu + row(j0 + r))[ic];
      bv[r] = (mv + row(j0 + r))[ic];
    }
  }
  auto m = [](int b) -> T { return MASKED ? (b ? T(1) : T(0)) : T(1); };
  // Vorticity at the X points and the averaged velocities there (rows j0 - 1 ..
  // j0 + R - 1), kinetic energy at the T points (rows j0 .. j0 + R).
  T ve[R + 1], uw[R + 1], z[R + 1], vq[ENS ? R + 1 : 1], uq[ENS ? R + 1 : 1], K[R + 1];
#pragma unroll
  for (int r = 0; r < R + 1; ++r) {
    const T q = m(bq[MASKED ? r : 0]), h = m(bh[MASKED ? r : 0]);
    ve[r] = east(vc[r]);
    z[r] = ((ve[r] - vc[r]) * idx - (uc[r + 1] - uc[r]) * idy) * q;
    if constexpr (ENS) {
      vq[r] = T(0.5) * (vc[r] + ve[r]) * q;
      uq[r] = T(0.5) * (uc[r] + uc[r + 1]) * q;
    }
    uw[r] = west(uc[r + 1]);
    const T ut = T(0.5) * (uc[r + 1] + uw[r]) * h, vt = T(0.5) * (vc[r + 1] + vc[r]) * h;
    K[r] = T(0.5) * (ut * ut + vt * vt);
  }
  const bool lout = lane >= 1 && lane <= 62 && i < nx, col = i >= 2 && i <= nx - 3;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int j = j0 + r;
    const T mu0 = m(bu[MASKED ? r : 0]), mv0 = m(bv[MASKED ? r : 0]);
    const T z00 = z[r + 1], zS = z[r], zW = west(z00), K00 = K[r];
    const T dKdx = (east(K00) - K00) * idx * mu0;
    const T dKdy = (K[r + 1] - K00) * idy * mv0;
    T zvu = T(0), zuv = T(0);
    if constexpr (SCHEME == kEnergy || SCHEME == kArakawaLamb) {
      const T z_u = T(0.5) * (z00 + zS) * mu0;
      const T v_u = T(0.25) * (vc[r + 1] + vc[r] + ve[r + 1] + ve[r]) * mu0;
      const T z_v = T(0.5) * (z00 + zW) * mv0;
      const T u_v = T(0.25) * (uc[r + 1] + uc[r + 2] + uw[r] + uw[r + 1]) * mv0;
      zvu = z_u * v_u;
      zuv = z_v * u_v;
    }
    if constexpr (ENS) {
      const T zs_u = T(0.5) * (z00 * vq[r + 1] + zS * vq[r]) * mu0;
      const T zs_v = T(0.5) * (z00 * uq[r + 1] + zW * west(uq[r + 1])) * mv0;
      if constexpr (SCHEME == kEnstrophy) {
        zvu = zs_u;
        zuv = zs_v;
      } else {
        constexpr T a = T(1.0 / 3.0);
        zvu = a * zvu + (T(1) - a) * zs_u;
        zuv = a * zuv + (T(1) - a) * zs_v;
      }
    }
    if (lout && j < ny) {
      const bool in = col && j >= 2 && j <= ny - 3;
      (du + (int64_t)j * nx)[i] = in ? (zvu - dKdx) * mu0 : T(0);
      (dv + (int64_t)j * nx)[i] = in ? (-zuv - dKdy) * mv0 : T(0);
    }
  }
}

// Fields of kMomMany cells and more: 4 rows a wavefront, smaller ones 1 (more
// wavefronts, shorter chains: 500^2 masked FP64 3.9 us).
constexpr int64_t kMomMany = 1 << 19;

template <typename T>
int momentum(const T* u, const T* v, T* du, T* dv, int scheme, const uint8_t* mh,
             const uint8_t* mu, const uint8_t* mv, const uint8_t* mq, int ny, int nx, double dx,
             double dy, hipStream_t s) {
  FVX_CHECK_ARG(u && v && du && dv, "null field pointer");
  FVX_CHECK_ARG(ny >= 3 && nx >= 3, "array too small (%d x %d)", ny, nx);
  FVX_CHECK_ARG(dx > 0 && dy > 0, "grid spacing must be positive");
  FVX_CHECK_ARG(scheme >= 0 && scheme <= 2,
                "Unknown scheme %d: 0 energy, 1 enstrophy, 2 Arakawa-Lamb", scheme);
  const bool masked = mh || mu || mv || mq;
  FVX_CHECK_ARG(!masked || (mh && mu && mv && mq), "pass all four stagger masks or none");
  const bool many = (int64_t)ny * nx >= kMomMany;
  const int tx = cdiv(nx, kMomCols), nt = tx * cdiv(ny, many ? 4 : 1);
  const dim3 g(cdiv(nt, 4)), b(256);
  const T ix = (T)(1.0 / dx), iy = (T)(1.0 / dy);
#define FVX_MOM(S, M)                                                                             \
  do {                                                                                           \
    if (many)                                                                                    \
      hipLaunchKernelGGL((momentum_kernel<T, S, M, 4>), g, b, 0, s, u, v, du, dv, mh, mu, mv, mq, \
                         ny, nx, ix, iy, tx, nt);                                                \
    else                                                                                         \
      hipLaunchKernelGGL((momentum_kernel<T, S, M, 1>), g, b, 0, s, u, v, du, dv, mh, mu, mv, mq, \
                         ny, nx, ix, iy, tx, nt);                                                \
  } while (0)
  if (masked) {
    if (scheme == kEnergy) FVX_MOM(kEnergy, true);
    else if (scheme == kEnstrophy) FVX_MOM(kEnstrophy, true);
    else FVX_MOM(kArakawaLamb, true);
  } else {
    if (scheme == kEnergy) FVX_MOM(kEnergy, false);
    else if (scheme == kEnstrophy) FVX_MOM(kEnstrophy, false);
    else FVX_MOM(kArakawaLamb, false);
  }
#undef FVX_MOM
  FVX_LAUNCH_CHECK();
  return kOk;
}

}  // namespace fvx

extern "C" {
int fvx_momentum_advection2d_f32(const float* u, const float* v, float* du, float* dv, int scheme,
                                 const uint8_t* mask_h, const uint8_t* mask_u,
                                 const uint8_t* mask_v, const uint8_t* mask_xy, int ny, int nx,
                                 double dx, double dy, void* stream) {
  return fvx::momentum<float>(u, v, du, dv, scheme, mask_h, mask_u, mask_v, mask_xy, ny, nx, dx,
                              dy, (hipStream_t)stream);
}
int fvx_momentum_advection2d_f64(const double* u, const double* v, double* du, double* dv,
                                 int scheme, const uint8_t* mask_h, const uint8_t* mask_u,
                                 const uint8_t* mask_v, const uint8_t* mask_xy, int ny, int nx,
                                 double dx, double dy, void* stream) {
  return fvx::momentum<double>(u, v, du, dv, scheme, mask_h, mask_u, mask_v, mask_xy, ny, nx, dx,
                               dy, (hipStream_t)stream);
}
}
