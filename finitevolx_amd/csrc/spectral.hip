// Spectral Helmholtz solvers (lap - lambda) psi = f on rectangles, the
// drop-in for solve_helmholtz_{dst,dct,fft} (re-exported from spectraldiffx
// v0.0.10 by solvers/spectral.py:14-128; used by scripts/qg_1p5_layer.py:443).
//
// Each transform diagonalises one of this library's 5-point operators
// exactly, so the solve is the operator's exact inverse:
//   dst : Dirichlet, zero just outside the array (DST-I; eigenvalues
//         -4/dx^2 sin^2(pi (k+1) / (2 (n+1))), dst1_eigenvalues)
//   dct : no-flux cell-centred Neumann (DCT-II / DCT-III pair; eigenvalues
//         -4/dx^2 sin^2(pi k / (2 n)); the k = l = 0 mode is set to zero
//         when the operator is singular)
//   fft : periodic (eigenvalues -4/dx^2 sin^2(pi k / n))
// DST / DCT plans of the sizes of use_gemm transform by matrix products on
// the FP64 matrix cores (spec_gemm_kernel: four launches for a whole batch of
// right-hand sides); others by batched real FFTs (hipFFT) of the odd /
// even extension of each row, written transposed so the y transform is again a
// batch of contiguous rows; periodic solves by hipFFT's 2-D real FFT.

#include <hipfft/hipfft.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

#include "fvx_common.hpp"

namespace fvx {

enum SpecBC : int { kDst = 0, kDct = 1, kFft = 2 };

template <typename T>
struct Cplx;
template <>
struct Cplx<double> {
  using type = hipfftDoubleComplex;
};
template <>
struct Cplx<float> {
  using type = hipfftComplex;
};

// Row r of src (length n, pitch ld) -> extended real row of length M.
template <typename T>
__global__ void ext_build_kernel(const T* __restrict__ src, int64_t ld, T* __restrict__ ext,
                                 int rows, int n, int M, int bc) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int r = blockIdx.y;
  if (k >= M || r >= rows) return;
  const T* x = src + (int64_t)r * ld;
  T v;
  if (bc == kDst) {  // [0, x0..x_{n-1}, 0, -x_{n-1}..-x0], M = 2(n+1)
    if (k == 0 || k == n + 1) v = T(0);
    else if (k <= n) v = x[k - 1];
    else v = -x[2 * n + 1 - k];
  } else {  // [x0..x_{n-1}, x_{n-1}..x0], M = 2n
    v = (k < n) ? x[k] : x[2 * n - 1 - k];
  }
  ext[(int64_t)r * M + k] = v;
}

// Spectrum row r (length M/2+1) -> transform coefficient k, written
// transposed: out[k * rows + r].
template <typename T, typename C>
__global__ void ext_extract_kernel(const C* __restrict__ spec, T* __restrict__ out, int rows,
                                   int n, int M, int bc) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int r = blockIdx.y;
  if (k >= n || r >= rows) return;
  const C* row = spec + (int64_t)r * (M / 2 + 1);
  T v;
  if (bc == kDst) {
    v = T(-0.5) * (T)row[k + 1].y;  // sum_j x_j sin(pi (k+1) (j+1) / (n+1))
  } else {
    const double th = -M_PI * k / (2.0 * n);
    const double c = cos(th), s = sin(th);
    v = (T)(0.5 * ((double)row[k].x * c - (double)row[k].y * s));  // DCT-II
  }
  out[(int64_t)k * rows + r] = v;
}

// DCT-III via C2R: V_k = X_k e^{i pi k / 2n} (k < n), V_n = 0.
template <typename T, typename C>
__global__ void dct3_build_kernel(const T* __restrict__ X, C* __restrict__ V, int rows, int n) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int r = blockIdx.y;
  if (k > n || r >= rows) return;
  C v;
  if (k == n) {
    v.x = 0;
    v.y = 0;
  } else {
    const double th = M_PI * k / (2.0 * n);
    const double x = (double)X[(int64_t)r * n + k];
    v.x = (T)(x * cos(th));
    v.y = (T)(x * sin(th));
  }
  V[(int64_t)r * (n + 1) + k] = v;
}

// First n samples of each length-2n C2R row, scaled, written transposed.
template <typename T>
__global__ void dct3_extract_kernel(const T* __restrict__ v, T* __restrict__ out, int rows, int n,
                                    T scale) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int r = blockIdx.y;
  if (k >= n || r >= rows) return;
  out[(int64_t)k * rows + r] = v[(int64_t)r * 2 * n + k] * scale;
}

// Divide the (nx, ny)-transposed coefficients by the operator eigenvalues.
template <typename T>
__global__ void eig_divide_kernel(T* __restrict__ c, int nx, int ny, int bc, double dx, double dy,
                                  double lam, double scale) {
  const int l = blockIdx.x * blockDim.x + threadIdx.x;  // y index (fast)
  const int k = blockIdx.y;                             // x index
  if (l >= ny || k >= nx) return;
  double ex, ey;
  if (bc == kDst) {
    const double sx = sin(M_PI * (k + 1) / (2.0 * (nx + 1))), sy = sin(M_PI * (l + 1) / (2.0 * (ny + 1)));
    ex = -4.0 / (dx * dx) * sx * sx;
    ey = -4.0 / (dy * dy) * sy * sy;
  } else {
    const double sx = sin(M_PI * k / (2.0 * nx)), sy = sin(M_PI * l / (2.0 * ny));
    ex = -4.0 / (dx * dx) * sx * sx;
    ey = -4.0 / (dy * dy) * sy * sy;
  }
  const double d = ex + ey - lam;
  const int64_t i = (int64_t)k * ny + l;
  c[i] = (d != 0.0) ? (T)((double)c[i] * scale / d) : T(0);
}

template <typename C>
__global__ void fft_divide_kernel(C* __restrict__ c, int ny, int nx, double dx, double dy,
                                  double lam, double scale) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;  // x wavenumber, 0..nx/2
  const int l = blockIdx.y;                             // y wavenumber, 0..ny-1
  const int nk = nx / 2 + 1;
  if (k >= nk || l >= ny) return;
  const double sx = sin(M_PI * k / nx), sy = sin(M_PI * l / ny);
  const double d = -4.0 / (dx * dx) * sx * sx - 4.0 / (dy * dy) * sy * sy - lam;
  C& v = c[(int64_t)l * nk + k];
  const double f = (d != 0.0) ? scale / d : 0.0;
  v.x = v.x * f;
  v.y = v.y * f;
}

template <typename T>
struct FftTypes;
template <>
struct FftTypes<double> {
  static constexpr hipfftType r2c = HIPFFT_D2Z, c2r = HIPFFT_Z2D;
  static hipfftResult fwd(hipfftHandle p, double* i, hipfftDoubleComplex* o) {
    return hipfftExecD2Z(p, i, o);
  }
  static hipfftResult inv(hipfftHandle p, hipfftDoubleComplex* i, double* o) {
    return hipfftExecZ2D(p, i, o);
  }
};
template <>
struct FftTypes<float> {
  static constexpr hipfftType r2c = HIPFFT_R2C, c2r = HIPFFT_C2R;
  static hipfftResult fwd(hipfftHandle p, float* i, hipfftComplex* o) {
    return hipfftExecR2C(p, i, o);
  }
  static hipfftResult inv(hipfftHandle p, hipfftComplex* i, float* o) {
    return hipfftExecC2R(p, i, o);
  }
};

// ---------------------------------------------------------------------------
// Transforms as matrix products.
//
// The kernels sin(pi (j + 1) (k + 1) / (n + 1)) and cos(pi (2 j + 1) k / 2 n)
// are even (k even) or odd (k odd) under j -> n - 1 - j, so a forward
// transform contracts x_j + x_{n-1-j} with the h x n0 matrix of the even k
// (class 0) and x_j - x_{n-1-j} with the h x n1 matrix of the odd ones (class
// 1; h = n0 = ceil(n / 2), n1 = floor(n / 2)), and the inverse one gives
// x_j = E_j + O_j, x_{n-1-j} = E_j - O_j: half the products of the full
// matrix.  Spectral indices stay ordered by class.
//
// Why: for the extended lengths 2 (n + 1) hipFFT falls to Bluestein's method
// at most n (n = 512: 1026 = 2 3^3 19), and each transform took an extension,
// 3-4 FFT kernels and an extraction per right-hand side.  Arithmetic is FP64
// for both precisions, each sum in chunks of 16 products.  Bound: the chain of a
// slab (two barriers, staging, both operands of every matrix instruction from
// LDS): the matrix cores are busy 0.20 to 0.28 of the time, the VALU 0.13 to
// 0.25, the memory 0.1 (v_mfma_f64_16x16x4 alone reaches 45 TFLOP/s; 64 TFLOP/s
// of plain FMAs would need four times the LDS reads).  Measured: 3 x 512 x 768
// DST 149 us a solve (20 TFLOP/s) against 535 through hipFFT; error against long double
// 3.2e-16 to 4.4e-16 (FP32 data 3.6e-8 to 6.1e-8) from 64 to 512 points, hipFFT
// 3.1e-16 to 7.6e-16 (1.4e-7 to 3.1e-7).
// ---------------------------------------------------------------------------
constexpr int kSpecBatch = 16;  // right-hand sides a launch

// Whether an extended length has a direct FFT (hipFFT's radices).
static bool fft_smooth(int m) {
  for (int p : {2, 3, 5, 7, 11, 13})
    while (m % p == 0) m /= p;
  return m == 1;
}
// Whether a plan transforms by matrix products: where they take less time than
// the FFTs did, by the two estimates below (us of a solve of one slice).  They
// fit 451 shapes of 2 to 3000 points an axis, each timed both ways: the products
// within 8% (FP64; 13% FP32) rms, the FFTs within 15%; the route took at most 1.2
// times the faster one's time (1.4 with an axis of 2 points), a rule on ny + nx
// alone up to 1.7.  Measured, products / FFTs:
//            FP64                         FP32
//   DCT  500 x  900    76 / 103      500 x 500    64 /  73     (direct lengths)
//        800 x  900   150 / 133      128 x 1100   81 /  69
//   DST  500 x  900    76 / 165      500 x 900    96 / 133     (others)
//       1023 x 1800   449 / 349     1023 x 1100  299 / 186
//         64 x 2900   135 / 158       64 x 1800  116 /  78
static double products_us(int ny, int nx, int bits) {
  double slabs = 0, second = 0, rounds = 0;  // of 64 points: all, > 256 blocks, > 512
  const auto launch = [&](int k, int blocks) {
    slabs += k;
    second += blocks > 256 ? k : 0;
    rounds += (double)k * (cdiv(blocks, 512) - 1);
  };
  const auto axis = [&](int n, int other) {
    const int h = (n + 1) / 2, n1 = n / 2, o = cdiv(other, 32);
    launch(cdiv(h, 64), o * (cdiv(h, 32) + cdiv(n1, 32)));
    launch(cdiv(h, 64) + cdiv(n1, 64), o * cdiv(h, 32));
  };
  axis(nx, ny);
  axis(ny, nx);
  const double cells = (double)ny * nx;
  return bits == 64 ? 9.3 + 1.43 * slabs + 0.4 * second + 1.78 * rounds + 4.24e-5 * cells
                    : 10.8 + 1.71 * slabs + 1.76 * rounds + 7.58e-5 * cells;
}
static double ffts_us(int ny, int nx, int slow, int bits) {
  // by the axes without a direct FFT (none, one, two; the last two again with an
  // axis over 2047 points): us, ns a cell
  static const double cost[2][5][2] = {
      {{53, 0.101}, {68, 0.132}, {82, 0.2}, {115, 0.184}, {131, 0.206}},  // FP64
      {{57, 0.06}, {68, 0.085}, {81, 0.13}, {95, 0.089}, {100, 0.13}}};   // FP32
  const double* c = cost[bits == 64 ? 0 : 1][slow + (slow && std::max(ny, nx) > 2047 ? 2 : 0)];
  return c[0] + 1e-3 * c[1] * ny * nx;
}
static bool use_gemm(int ny, int nx, int bc, int bits) {
  if (bc == kFft) return false;
  const int ext = bc == kDst ? 2 : 0;
  const int slow = !fft_smooth(2 * nx + ext) + !fft_smooth(2 * ny + ext);
  // (nothing beyond these sums was timed)
  const int most = bits == 64 ? (slow ? 3072 : 1800) : (slow ? 2200 : 1400);
  return ny + nx <= most && products_us(ny, nx, bits) <= ffts_us(ny, nx, slow, bits);
}
typedef double f64x4 __attribute__((ext_vector_type(4)));

template <typename T>
struct SpecGemm {
  const T* in;   // forward: physical along the transformed axis, else spectral
  T* out;
  int64_t ld_in, bs_in, ld_out, bs_out;  // row pitch and batch stride
  const double *s0, *s1;  // class matrices [h][n0], [h][n1]
  int n, h, n0, n1;       // the transformed axis
  int other;              // points along the other axis
  // Division by the eigenvalues (forward, second axis): squared sines of this
  // axis and the other in spectral order.
  const double *et, *eo;
  double ct, co, scale;
  int divide, halve0;  // halve0: the DCT's k = 0 weight along each axis
  int ring;            // (last product) zero the one-cell ring around the output
  double lam[kSpecBatch];
};

// LEFT: the transformed axis is the arrays' row index (out = S in), else the
// column index (out = in S).  A workgroup owns 32 outputs x 32 points of the
// other axis; its 8 waves are two groups that split each K slab (64 points)
// between them, four waves of 16 x 16 outputs in a group, and sum their parts
// through LDS at the end.  Small tiles and two groups keep several short
// chains on every CU: 3 x 512 x 768 takes 143 us a solve (151 with the chunked
// sums), 156 with tiles of 64, 167 with four groups.
constexpr int kSpecThreads = 512;
// The cells of the one-cell zero ring that lie next to cell (j, i) of the
// ny x nx array at out.
template <typename T>
__device__ __forceinline__ void ring_around(T* out, int64_t ld, int j, int i, int ny, int nx) {
  T* p = out + (int64_t)j * ld + i;
  const bool w = i == 0, e = i == nx - 1;
  if (w) p[-1] = T(0);
  if (e) p[1] = T(0);
  if (j == 0) {
    p[-ld] = T(0);
    if (w) p[-ld - 1] = T(0);
    if (e) p[-ld + 1] = T(0);
  }
  if (j == ny - 1) {
    p[ld] = T(0);
    if (w) p[ld - 1] = T(0);
    if (e) p[ld + 1] = T(0);
  }
}
template <typename T, bool LEFT, bool INV>
__global__ __launch_bounds__(kSpecThreads) void spec_gemm_kernel(SpecGemm<T> g) {
  constexpr int BT = 32, BK = 64, P = BT + 2, PER = BT * BK / kSpecThreads;
  constexpr int NC = INV ? 2 : 1;  // accumulated classes
  __shared__ __align__(16) double smem[2 * BK * P];
  double(*sm)[P] = reinterpret_cast<double(*)[P]>(smem);           // matrix operand [k][t]
  double(*sd)[P] = reinterpret_cast<double(*)[P]>(smem + BK * P);  // data operand [k][o]
  static_assert(NC * 4 * 256 <= 2 * BK * P, "a group's sums fit in the slabs");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2, w4 = wave & 3;
  const int o0 = blockIdx.x * BT;
  int cls = 0, t0 = blockIdx.y * BT;
  if constexpr (!INV) {
    const int tiles0 = (g.n0 + BT - 1) / BT;
    if ((int)blockIdx.y >= tiles0) {
      cls = 1;
      t0 = (blockIdx.y - tiles0) * BT;
    }
  }
  const T* in = g.in + (int64_t)blockIdx.z * g.bs_in;
  const int nt = INV ? g.h : (cls ? g.n1 : g.n0);  // outputs of the class
  f64x4 acc[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] = f64x4{0., 0., 0., 0.};

  // Element e of a slab: its place (contiguous in memory along the fast index).
  auto mat_at = [&](int e, int& k, int& t) {
    if constexpr (INV) {
      k = e % BK;
      t = e / BK;
    } else {
      t = e % BT;
      k = e / BT;
    }
  };
  auto dat_at = [&](int e, int& k, int& o) {
    if constexpr (LEFT) {
      o = e % BT;
      k = e / BT;
    } else {
      k = e % BK;
      o = e / BK;
    }
  };
  double rm[PER], rd[PER];
  auto load = [&](int c, int k0) {
    const double* S = c ? g.s1 : g.s0;
    const int nc = c ? g.n1 : g.n0, K = INV ? nc : g.h;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      int k, t;
      mat_at(tid + i * kSpecThreads, k, t);
      k += k0;
      t += t0;
      rm[i] = (k < K && t < nt) ? S[INV ? (int64_t)t * nc + k : (int64_t)k * nc + t] : 0.0;
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      int k, o;
      dat_at(tid + i * kSpecThreads, k, o);
      k += k0;
      o += o0;
      double v = 0.0;
      if (k < K && o < g.other) {
        auto at = [&](int q) -> double {
          return (double)in[LEFT ? (int64_t)q * g.ld_in + o : (int64_t)o * g.ld_in + q];
        };
        if constexpr (INV) {
          v = at((c ? g.n0 : 0) + k);
        } else {
          const int km = g.n - 1 - k;
          const double u = at(k), w = at(km);
          v = c ? u - w : u + w;
          if (km == k) v = c ? 0.0 : u;  // (the middle point has no partner)
        }
      }
      rd[i] = v;
    }
  };
  const int lr = lane & 15, lk = lane >> 4;
  const int wm = (w4 >> 1) * 16, wn = (w4 & 1) * 16;  // rows / columns of D
#pragma unroll
  for (int ci = 0; ci < NC; ++ci) {
    const int c = INV ? ci : cls;
    const int K = INV ? (c ? g.n1 : g.n0) : g.h;
    load(c, 0);
    for (int k0 = 0; k0 < K; k0 += BK) {
      __syncthreads();  // (the previous slab has been read)
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        int k, t;
        mat_at(tid + i * kSpecThreads, k, t);
        sm[k][t] = rm[i];
        dat_at(tid + i * kSpecThreads, k, t);
        sd[k][t] = rd[i];
      }
      __syncthreads();
      if (k0 + BK < K) load(c, k0 + BK);
      // chunks of 16 products, summed on their own: a serial sum of the whole
      // axis rounds sqrt(n / 16) times as much
      f64x4 chunk[2] = {f64x4{0., 0., 0., 0.}, f64x4{0., 0., 0., 0.}};
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k = grp * 32 + h * 16 + 4 * kk + lk;
          const double fa = (LEFT ? sm : sd)[k][wm + lr], fb = (LEFT ? sd : sm)[k][wn + lr];
          chunk[h] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa, fb, chunk[h], 0, 0, 0);
        }
      acc[ci] += chunk[0] + chunk[1];
    }
  }
  // The second group's sums into the first's.
  f64x4* part = reinterpret_cast<f64x4*>(smem) + w4 * 64 + lane;
  __syncthreads();
  if (grp == 1) {
#pragma unroll
    for (int c = 0; c < NC; ++c) part[c * 256] = acc[c];
  }
  __syncthreads();
  if (grp == 1) return;
#pragma unroll
  for (int c = 0; c < NC; ++c) acc[c] += part[c * 256];

  // D of a 16 x 16 block: row 4 i + lane / 16, column lane % 16.
  T* out = g.out + (int64_t)blockIdx.z * g.bs_out;
  const double lam = g.lam[blockIdx.z];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = wm + 4 * i + lk, n = wn + lr;
    const int t = t0 + (LEFT ? m : n), o = o0 + (LEFT ? n : m);
    if (t >= nt || o >= g.other) continue;
    auto put_at = [&](int q, double v) {
      out[LEFT ? (int64_t)q * g.ld_out + o : (int64_t)o * g.ld_out + q] = (T)v;
      if constexpr (INV && !LEFT) {
        if (g.ring) ring_around(out, g.ld_out, o, q, g.other, g.n);
      }
    };
    if constexpr (INV) {
      const double e = acc[0][i], d = acc[NC - 1][i];
      put_at(t, e + d);
      if (g.n - 1 - t != t) put_at(g.n - 1 - t, e - d);
    } else {
      const int q = (cls ? g.n0 : 0) + t;
      double v = acc[0][i];
      if (g.divide) {
        const double den = g.ct * g.et[q] + g.co * g.eo[o] - lam;
        double f = g.scale;
        if (g.halve0) f *= (q == 0 ? 0.5 : 1.0) * (o == 0 ? 0.5 : 1.0);
        v = den != 0.0 ? v * f / den : 0.0;
      }
      put_at(q, v);
    }
  }
}

// Class matrices and squared sines of one axis of n points.
__global__ void spec_matrix_kernel(double* __restrict__ s0, double* __restrict__ s1,
                                   double* __restrict__ e, int n, int bc) {
  const int h = (n + 1) / 2, n0 = h, n1 = n / 2;
  const int64_t total = (int64_t)h * n;
  for (int64_t x = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; x < total;
       x += (int64_t)gridDim.x * blockDim.x) {
    const int j = (int)(x / n), q = (int)(x % n);
    const int c = q >= n0, r = c ? q - n0 : q, k = 2 * r + c;
    // the angle as an integer multiple of pi / n', reduced exactly
    double v;
    if (bc == kDst) {
      const int64_t m = ((int64_t)(j + 1) * (k + 1)) % (2 * (n + 1));
      v = sinpi((double)m / (n + 1));
    } else {
      const int64_t m = ((int64_t)(2 * j + 1) * k) % (4 * n);
      v = cospi((double)m / (2.0 * n));
    }
    (c ? s1 : s0)[(int64_t)j * (c ? n1 : n0) + r] = v;
    if (j == 0) {
      const double sn = bc == kDst ? sinpi((k + 1) / (2.0 * (n + 1))) : sinpi(k / (2.0 * n));
      e[q] = sn * sn;
    }
  }
}

struct SpecAxis {
  int n = 0;
  double *s0 = nullptr, *s1 = nullptr, *e = nullptr;  // one allocation, s0
};

struct SpecPlan {
  int ny, nx, bc, prec;
  // per-direction batched 1-D plans (x: ny rows of length Mx; y: nx rows of length My)
  hipfftHandle fx = 0, fy = 0, ix = 0, iy = 0, f2 = 0, i2 = 0;
  void* ext = nullptr;   // real extension buffer
  void* spec = nullptr;  // complex buffer
  void* a = nullptr;     // transposed real (nx, ny)
  void* b = nullptr;     // real (ny, nx) / second transposed buffer
  bool gemm = false;     // transforms by matrix products
  SpecAxis ax, ay;
  // Calls that work in the plan's own buffers (and hipFFT's, behind its handles)
  // are enqueued one at a time, each after the last one's end (SpecUse).
  std::mutex mu;
  hipEvent_t last = nullptr;  // the end of the last use, once ``shared``
  hipStream_t owner = nullptr;  // the stream of every use so far, until then
  bool used = false, shared = false;
};

// One use of a plan's own buffers on stream ``s``.  Calls from several threads
// and streams share the plan, so a use waits for the event behind the last one,
// on the device; the host does not wait.  A plan that one stream alone has used
// needs no event (each costs 3.5 us on the device: 21 us a periodic solve of 64^2
// without, 25 with).  Under capture there is nothing to wait on (an event from
// outside may not enter a graph): the program orders a graph's replays with other
// uses of the plan.
struct SpecUse {
  SpecPlan* P;
  hipStream_t s;
  std::unique_lock<std::mutex> lock;
  bool eager = false;
  int rc = kOk;
  static bool capturing(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) == hipSuccess) return st != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return true;
  }
  SpecUse(SpecPlan* P_, hipStream_t s_) : P(P_), s(s_), lock(P_->mu), eager(!capturing(s_)) {
    if (!eager || !P->used || (!P->shared && s == P->owner)) return;
    const bool event = P->shared || (!capturing(P->owner) &&
                                     hipEventRecord(P->last, P->owner) == hipSuccess);
    P->shared = true;
    if (event && hipStreamWaitEvent(s, P->last, 0) == hipSuccess) return;
    // (the owner may be gone, or part of a capture by now)
    (void)hipGetLastError();
    if (hipDeviceSynchronize() == hipSuccess) return;
    set_error("could not order the solve behind the plan's last one");
    rc = kHipError;
  }
  // After the enqueue (also a failed one: some of it may run); its status, or
  // this one's.
  int end(int enqueued) {
    if (!eager || rc) return enqueued;
    P->used = true;
    P->owner = s;
    if (!P->shared || hipEventRecord(P->last, s) == hipSuccess) return enqueued;
    set_error("could not record the end of the solve");
    return kHipError;
  }
};

#define FVX_FFT(call)                                                  \
  do {                                                                 \
    hipfftResult r_ = (call);                                          \
    if (r_ != HIPFFT_SUCCESS) {                                        \
      ::fvx::set_error("hipFFT error %d at %s:%d", (int)r_, __FILE__, __LINE__); \
      return ::fvx::kHipError;                                         \
    }                                                                  \
  } while (0)

static int spec_axis(SpecAxis& A, int n, int bc) {
  A.n = n;
  const size_t h = (n + 1) / 2, n1 = n / 2;
  FVX_HIP(hipMalloc(&A.s0, (h * h + h * n1 + n) * sizeof(double)));
  A.s1 = A.s0 + h * h;
  A.e = A.s1 + h * n1;
  hipLaunchKernelGGL(spec_matrix_kernel, dim3(1024), dim3(256), 0, nullptr, A.s0, A.s1, A.e, n, bc);
  FVX_LAUNCH_CHECK();
  FVX_HIP(hipStreamSynchronize(nullptr));  // solves run on any stream
  return kOk;
}

template <typename T>
static int spec_create(SpecPlan* P) {
  const int ny = P->ny, nx = P->nx;
  if (use_gemm(ny, nx, P->bc, P->prec)) {
    P->gemm = true;
    FVX_HIP(hipMalloc(&P->a, 2 * (size_t)ny * nx * sizeof(T)));
    if (int rc = spec_axis(P->ax, nx, P->bc)) return rc;
    return spec_axis(P->ay, ny, P->bc);
  }
  using FT = FftTypes<T>;
  using C = typename Cplx<T>::type;
  size_t ext_elems = 0, spec_elems = 0;
  if (P->bc == kFft) {
    FVX_FFT(hipfftPlan2d(&P->f2, ny, nx, FT::r2c));
    FVX_FFT(hipfftPlan2d(&P->i2, ny, nx, FT::c2r));
    spec_elems = (size_t)ny * (nx / 2 + 1);
  } else {
    const int Mx = P->bc == kDst ? 2 * (nx + 1) : 2 * nx;
    const int My = P->bc == kDst ? 2 * (ny + 1) : 2 * ny;
    FVX_FFT(hipfftPlan1d(&P->fx, Mx, FT::r2c, ny));
    FVX_FFT(hipfftPlan1d(&P->fy, My, FT::r2c, nx));
    if (P->bc == kDct) {
      FVX_FFT(hipfftPlan1d(&P->ix, 2 * nx, FT::c2r, ny));
      FVX_FFT(hipfftPlan1d(&P->iy, 2 * ny, FT::c2r, nx));
    }
    ext_elems = std::max((size_t)ny * Mx, (size_t)nx * My);
    spec_elems = std::max((size_t)ny * (Mx / 2 + 1), (size_t)nx * (My / 2 + 1));
  }
  const size_t N = (size_t)ny * nx;
  FVX_HIP(hipMalloc(&P->spec, spec_elems * sizeof(C)));
  if (ext_elems) FVX_HIP(hipMalloc(&P->ext, ext_elems * sizeof(T)));
  FVX_HIP(hipMalloc(&P->a, N * sizeof(T)));
  FVX_HIP(hipMalloc(&P->b, N * sizeof(T)));
  return kOk;
}

// Forward sine/cosine transform of `rows` rows of length n (pitch ld) ->
// transposed coefficients (n, rows) in out.
template <typename T>
static int fwd_rows(SpecPlan* P, hipfftHandle plan, const T* src, int64_t ld, int rows, int n,
                    T* out, hipStream_t s) {
  using C = typename Cplx<T>::type;
  const int M = P->bc == kDst ? 2 * (n + 1) : 2 * n;
  hipLaunchKernelGGL(ext_build_kernel<T>, dim3(cdiv(M, 256), rows), dim3(256), 0, s, src, ld,
                     (T*)P->ext, rows, n, M, P->bc);
  FVX_FFT(hipfftSetStream(plan, s));
  FVX_FFT(FftTypes<T>::fwd(plan, (T*)P->ext, (C*)P->spec));
  hipLaunchKernelGGL((ext_extract_kernel<T, C>), dim3(cdiv(n, 256), rows), dim3(256), 0, s,
                     (const C*)P->spec, out, rows, n, M, P->bc);
  FVX_LAUNCH_CHECK();
  return kOk;
}

// Inverse along rows (DST-I is its own inverse up to 2/(n+1); DCT-III via
// C2R): coefficients (rows, n) -> transposed values (n, rows), scaled.
template <typename T>
static int inv_rows(SpecPlan* P, hipfftHandle fplan, hipfftHandle iplan, const T* src, int rows,
                    int n, T* out, hipStream_t s) {
  using C = typename Cplx<T>::type;
  if (P->bc == kDst) {
    int rc = fwd_rows<T>(P, fplan, src, n, rows, n, out, s);
    return rc;  // scale folded into the eigenvalue division
  }
  hipLaunchKernelGGL((dct3_build_kernel<T, C>), dim3(cdiv(n + 1, 256), rows), dim3(256), 0, s,
                     src, (C*)P->spec, rows, n);
  FVX_FFT(hipfftSetStream(iplan, s));
  FVX_FFT(FftTypes<T>::inv(iplan, (C*)P->spec, (T*)P->ext));
  hipLaunchKernelGGL(dct3_extract_kernel<T>, dim3(cdiv(n, 256), rows), dim3(256), 0, s,
                     (const T*)P->ext, out, rows, n, (T)(1.0 / n));
  FVX_LAUNCH_CHECK();
  return kOk;
}

template <typename T>
__global__ void copy_pitched_kernel(const T* __restrict__ src, int64_t lds, T* __restrict__ dst,
                                    int64_t ldd, int ny, int nx) {
  const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
  if (i < nx && j < ny) dst[(int64_t)j * ldd + i] = src[(int64_t)j * lds + i];
}

template <typename T>
__global__ void ring_kernel(T* out, int64_t ld, int ny, int nx) {
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k < nx) {
    ring_around(out, ld, 0, k, ny, nx);
    ring_around(out, ld, ny - 1, k, ny, nx);
  }
  if (k < ny) {
    ring_around(out, ld, k, 0, ny, nx);
    ring_around(out, ld, k, nx - 1, ny, nx);
  }
}

template <typename T, bool LEFT, bool INV>
static int launch_spec(const SpecGemm<T>& g, int nb, hipStream_t s) {
  const dim3 grid(cdiv(g.other, 32), INV ? cdiv(g.h, 32) : cdiv(g.n0, 32) + cdiv(g.n1, 32), nb);
  hipLaunchKernelGGL((spec_gemm_kernel<T, LEFT, INV>), grid, dim3(kSpecThreads), 0, s, g);
  FVX_LAUNCH_CHECK();
  return kOk;
}

// Scratch of a batched solve: two fields a slice of one launch; the FFTs have
// theirs in the plan.
static int64_t work_elements(const SpecPlan* P, int nb) {
  return P->gemm ? (int64_t)2 * std::min(nb, kSpecBatch) * P->ny * P->nx : 0;
}

// nb solves (right-hand side b at rhs + b bs_rhs, solution at out + b bs_out,
// its lambda in lam[b]) by matrix products; work: work_elements(P, nb).
template <typename T>
static int gemm_solve(SpecPlan* P, const T* rhs, int64_t ld_rhs, int64_t bs_rhs, T* out,
                      int64_t ld_out, int64_t bs_out, int nb, const double* lam, double dx,
                      double dy, T* work, hipStream_t s, bool ring = false) {
  const int ny = P->ny, nx = P->nx;
  const int64_t N = (int64_t)ny * nx;
  for (int b0 = 0; b0 < nb; b0 += kSpecBatch) {
    const int m = std::min(kSpecBatch, nb - b0);
    T *A = work, *B = A + m * N;  // (the launches before have read theirs)
    SpecGemm<T> g;
    std::memset(&g, 0, sizeof(g));
    for (int b = 0; b < m; ++b) g.lam[b] = lam[b0 + b];
    auto axis = [&](const SpecAxis& X, int other) {
      g.n = X.n;
      g.h = g.n0 = (X.n + 1) / 2;
      g.n1 = X.n / 2;
      g.s0 = X.s0;
      g.s1 = X.s1;
      g.other = other;
    };
    auto arrays = [&](const T* in, int64_t ldi, int64_t bsi, T* o, int64_t ldo, int64_t bso) {
      g.in = in;
      g.ld_in = ldi;
      g.bs_in = bsi;
      g.out = o;
      g.ld_out = ldo;
      g.bs_out = bso;
    };
    axis(P->ax, ny);
    arrays(rhs + b0 * bs_rhs, ld_rhs, bs_rhs, A, nx, N);
    if (int rc = launch_spec<T, false, false>(g, m, s)) return rc;
    axis(P->ay, nx);
    arrays(A, nx, N, B, nx, N);
    g.divide = 1;
    g.halve0 = P->bc == kDct;
    g.et = P->ay.e;
    g.eo = P->ax.e;
    g.ct = -4.0 / (dy * dy);
    g.co = -4.0 / (dx * dx);
    g.scale = P->bc == kDst ? (2.0 / (nx + 1)) * (2.0 / (ny + 1)) : (2.0 / nx) * (2.0 / ny);
    if (int rc = launch_spec<T, true, false>(g, m, s)) return rc;
    g.divide = 0;
    arrays(B, nx, N, A, nx, N);
    if (int rc = launch_spec<T, true, true>(g, m, s)) return rc;
    axis(P->ax, ny);
    arrays(A, nx, N, out + b0 * bs_out, ld_out, bs_out);
    g.ring = ring;
    if (int rc = launch_spec<T, false, true>(g, m, s)) return rc;
  }
  return kOk;
}

template <typename T>
static int spec_solve(SpecPlan* P, const T* rhs, int64_t ld_rhs, T* out, int64_t ld_out,
                      double dx, double dy, double lam, hipStream_t s) {
  using C = typename Cplx<T>::type;
  const int ny = P->ny, nx = P->nx;
  if (P->gemm)
    return gemm_solve<T>(P, rhs, ld_rhs, 0, out, ld_out, 0, 1, &lam, dx, dy, (T*)P->a, s);
  T* A = (T*)P->a;
  T* B = (T*)P->b;
  if (P->bc == kFft) {
    hipLaunchKernelGGL(copy_pitched_kernel<T>, dim3(cdiv(nx, 64), cdiv(ny, 4)), dim3(64, 4), 0, s,
                       rhs, ld_rhs, A, (int64_t)nx, ny, nx);
    FVX_FFT(hipfftSetStream(P->f2, s));
    FVX_FFT(FftTypes<T>::fwd(P->f2, A, (C*)P->spec));
    hipLaunchKernelGGL((fft_divide_kernel<C>), dim3(cdiv(nx / 2 + 1, 256), ny), dim3(256), 0, s,
                       (C*)P->spec, ny, nx, dx, dy, lam, 1.0 / ((double)nx * ny));
    FVX_FFT(hipfftSetStream(P->i2, s));
    FVX_FFT(FftTypes<T>::inv(P->i2, (C*)P->spec, B));
    hipLaunchKernelGGL(copy_pitched_kernel<T>, dim3(cdiv(nx, 64), cdiv(ny, 4)), dim3(64, 4), 0, s,
                       B, (int64_t)nx, out, ld_out, ny, nx);
    FVX_LAUNCH_CHECK();
    return kOk;
  }
  // x transform of the ny rows -> A (nx, ny); y transform of the nx rows -> B (ny, nx)
  int rc = fwd_rows<T>(P, P->fx, rhs, ld_rhs, ny, nx, A, s);
  if (!rc) rc = fwd_rows<T>(P, P->fy, A, ny, nx, ny, B, s);
  if (rc) return rc;
  // B is (ny, nx) in (l, k) order; divide with the eigenvalues (B viewed as
  // (ny rows of nx): index l * nx + k).  Reuse eig_divide with swapped roles.
  double scale = 1.0;
  if (P->bc == kDst) scale = (2.0 / (nx + 1)) * (2.0 / (ny + 1));
  hipLaunchKernelGGL(eig_divide_kernel<T>, dim3(cdiv(nx, 256), ny), dim3(256), 0, s, B, ny, nx,
                     P->bc, dy, dx, lam, scale);
  // inverse along y (rows of length ny of the (nx, ny) layout) and x.
  rc = inv_rows<T>(P, P->fx, P->ix, B, ny, nx, A, s);  // rows = ny (l), length nx (k) -> A (nx, ny)
  if (!rc) rc = inv_rows<T>(P, P->fy, P->iy, A, nx, ny, B, s);  // -> B (ny, nx)
  if (rc) return rc;
  hipLaunchKernelGGL(copy_pitched_kernel<T>, dim3(cdiv(nx, 64), cdiv(ny, 4)), dim3(64, 4), 0, s,
                     B, (int64_t)nx, out, ld_out, ny, nx);
  FVX_LAUNCH_CHECK();
  return kOk;
}

}  // namespace fvx

extern "C" {

int fvx_spectral_plan_destroy(void* plan);

// bc: 0 = DST-I (Dirichlet), 1 = DCT-II (Neumann), 2 = FFT (periodic);
// precision 32 or 64.  ny, nx: the array the solve runs on (interior only).
int fvx_spectral_plan_create(int ny, int nx, int bc, int precision, void** plan_out) {
  using namespace fvx;
  FVX_CHECK_ARG(plan_out, "null plan_out");
  FVX_CHECK_ARG(ny >= 2 && nx >= 2, "spectral solve needs at least 2 x 2");
  FVX_CHECK_ARG(bc >= 0 && bc <= 2, "bc must be 0 (dst), 1 (dct) or 2 (fft)");
  FVX_CHECK_ARG(precision == 32 || precision == 64, "precision must be 32 or 64");
  SpecPlan* P = new SpecPlan();
  P->ny = ny;
  P->nx = nx;
  P->bc = bc;
  P->prec = precision;
  int rc = precision == 64 ? spec_create<double>(P) : spec_create<float>(P);
  if (!rc && hipEventCreateWithFlags(&P->last, hipEventDisableTiming) != hipSuccess) {
    set_error("could not create the plan's event");
    rc = kHipError;
  }
  if (rc) {
    fvx_spectral_plan_destroy(P);
    return rc;
  }
  *plan_out = P;
  return kOk;
}

int fvx_spectral_plan_destroy(void* plan) {
  using namespace fvx;
  if (!plan) return kOk;
  SpecPlan* P = (SpecPlan*)plan;
  (void)hipDeviceSynchronize();
  if (P->last) (void)hipEventDestroy(P->last);
  for (hipfftHandle h : {P->fx, P->fy, P->ix, P->iy, P->f2, P->i2})
    if (h) hipfftDestroy(h);
  (void)hipFree(P->ax.s0);
  (void)hipFree(P->ay.s0);
  (void)hipFree(P->ext);
  (void)hipFree(P->spec);
  (void)hipFree(P->a);
  (void)hipFree(P->b);
  delete P;
  return kOk;
}

// (lap - lambda) out = rhs for the plan's boundary condition; rhs / out pitched.
int fvx_spectral_helmholtz_f64(void* plan, const double* rhs, int64_t ld_rhs, double* out,
                               int64_t ld_out, double dx, double dy, double lambda_,
                               void* stream) {
  using namespace fvx;
  FVX_CHECK_ARG(plan && rhs && out, "null argument");
  SpecPlan* P = (SpecPlan*)plan;
  FVX_CHECK_ARG(P->prec == 64, "plan was built for float32");
  FVX_CHECK_ARG(dx > 0 && dy > 0, "grid spacing must be positive");
  SpecUse use(P, (hipStream_t)stream);
  if (use.rc) return use.rc;
  return use.end(
      spec_solve<double>(P, rhs, ld_rhs, out, ld_out, dx, dy, lambda_, (hipStream_t)stream));
}
int fvx_spectral_helmholtz_f32(void* plan, const float* rhs, int64_t ld_rhs, float* out,
                               int64_t ld_out, double dx, double dy, double lambda_,
                               void* stream) {
  using namespace fvx;
  FVX_CHECK_ARG(plan && rhs && out, "null argument");
  SpecPlan* P = (SpecPlan*)plan;
  FVX_CHECK_ARG(P->prec == 32, "plan was built for float64");
  FVX_CHECK_ARG(dx > 0 && dy > 0, "grid spacing must be positive");
  SpecUse use(P, (hipStream_t)stream);
  if (use.rc) return use.rc;
  return use.end(
      spec_solve<float>(P, rhs, ld_rhs, out, ld_out, dx, dy, lambda_, (hipStream_t)stream));
}

// Elements of the work array of a solve of nb slices.
int fvx_spectral_work_size(void* plan, int nb, int64_t* elements) {
  using namespace fvx;
  FVX_CHECK_ARG(plan && elements, "null argument");
  FVX_CHECK_ARG(nb >= 0, "negative batch");
  *elements = work_elements((SpecPlan*)plan, nb);
  return kOk;
}

// nb solves of contiguous (ny, nx) fields back to back, (lap - lambda_[b])
// out_b = rhs_b (lambda_: host array); out may be rhs.  work: device scratch of
// fvx_spectral_work_size elements for the call (the caller's, so that calls on
// several streams or threads do not share any); may be null where that is 0.
#define FVX_SPEC_BATCH(SUF, T, PREC)                                                             \
  int fvx_spectral_helmholtz_batch_##SUF(void* plan, const T* rhs, T* out, int nb,               \
                                         const double* lambda_, double dx, double dy, T* work,   \
                                         void* stream) {                                         \
    using namespace fvx;                                                                         \
    FVX_CHECK_ARG(plan, "null argument");                                                        \
    SpecPlan* P = (SpecPlan*)plan;                                                               \
    FVX_CHECK_ARG(P->prec == PREC, "plan was built for the other precision");                    \
    FVX_CHECK_ARG(dx > 0 && dy > 0, "grid spacing must be positive");                            \
    FVX_CHECK_ARG(nb >= 0, "negative batch");                                                    \
    if (nb == 0) return kOk; /* (an empty array has no address) */                               \
    FVX_CHECK_ARG(rhs && out && lambda_, "null argument");                                       \
    const int64_t N = (int64_t)P->ny * P->nx;                                                    \
    if (P->gemm) {                                                                               \
      FVX_CHECK_ARG(work, "null work array");                                                    \
      return gemm_solve<T>(P, rhs, P->nx, N, out, P->nx, N, nb, lambda_, dx, dy, work,           \
                           (hipStream_t)stream);                                                 \
    }                                                                                            \
    SpecUse use(P, (hipStream_t)stream);                                                         \
    int rc = use.rc;                                                                             \
    for (int b = 0; b < nb && !rc; ++b)                                                          \
      rc = spec_solve<T>(P, rhs + b * N, P->nx, out + b * N, P->nx, dx, dy, lambda_[b],          \
                         (hipStream_t)stream);                                                   \
    return use.end(rc);                                                                          \
  }
FVX_SPEC_BATCH(f64, double, 64)
FVX_SPEC_BATCH(f32, float, 32)
#undef FVX_SPEC_BATCH

// One solve on the interior of full (ny + 2, nx + 2) fields: out's one-cell
// ring is written zero, rhs' ring is not read.  work as in the batched solve.
#define FVX_SPEC_FIELD(SUF, T, PREC)                                                             \
  int fvx_spectral_helmholtz_field_##SUF(void* plan, const T* rhs, T* out, double dx, double dy, \
                                         double lambda_, T* work, void* stream) {                \
    using namespace fvx;                                                                         \
    FVX_CHECK_ARG(plan && rhs && out, "null argument");                                          \
    FVX_CHECK_ARG(rhs != out, "out must be another array");                                      \
    SpecPlan* P = (SpecPlan*)plan;                                                               \
    FVX_CHECK_ARG(P->prec == PREC, "plan was built for the other precision");                    \
    FVX_CHECK_ARG(dx > 0 && dy > 0, "grid spacing must be positive");                            \
    const int64_t ld = P->nx + 2;                                                                \
    hipStream_t s = (hipStream_t)stream;                                                         \
    if (P->gemm) {                                                                               \
      FVX_CHECK_ARG(work, "null work array");                                                    \
      return gemm_solve<T>(P, rhs + ld + 1, ld, 0, out + ld + 1, ld, 0, 1, &lambda_, dx, dy,     \
                           work, s, true);                                                       \
    }                                                                                            \
    SpecUse use(P, s);                                                                           \
    if (use.rc) return use.rc;                                                                   \
    if (int rc = use.end(                                                                        \
            spec_solve<T>(P, rhs + ld + 1, ld, out + ld + 1, ld, dx, dy, lambda_, s)))           \
      return rc;                                                                                 \
    hipLaunchKernelGGL(ring_kernel<T>, dim3(cdiv(std::max(P->ny, P->nx), 256)), dim3(256), 0, s, \
                       out + ld + 1, ld, P->ny, P->nx);                                          \
    FVX_LAUNCH_CHECK();                                                                          \
    return kOk;                                                                                  \
  }
FVX_SPEC_FIELD(f64, double, 64)
FVX_SPEC_FIELD(f32, float, 32)
#undef FVX_SPEC_FIELD
}
