// Level descriptors, tile-kernel arguments and block reductions shared by the
// multigrid kernels (mg.hip: tiles and coarse levels; mg_strip.hpp: strips).
#pragma once

#include "fvx_common.hpp"
#include "mg.hpp"

namespace fvx {

enum MgKind : int { kNoflux = 0, kDirichlet = 1 };

template <typename T>
struct LevelDev {
  int ny, nx;
  T idx2, idy2, lam;
  T inv_d;                 // Dirichlet scalar 1/diag
  const uint8_t* mask;     // nullptr = all wet
  const T* cx;             // noflux face coefficients (nullptr for Dirichlet)
  const T* cy;
  const T* inv;            // noflux inverse diagonal
  T* u;                    // iterate (coarse levels: error)
  T* b;                    // right-hand side (coarse levels: restricted residual)
  T* t;                    // scratch of the level kernels: sweep chains, the up leg's result
  T* t2;
  T* t3;
  // Dirichlet coarse levels with the wall correction: each dry or outside
  // neighbour adds wall_g / h^2 to the diagonal (a ghost value wall_g u_c
  // instead of 0); 0 = off.
  T wall_g;
  // The mask packed by columns (with mask): word (blk, i) = the mask of rows
  // 32 blk .. 32 blk + 31 of column i as bits (rows beyond the level 0),
  // blocks 0 .. ny / 32 + 1, so a 64-bit window from any row block is valid.
  const uint32_t* mcol;
};

template <typename T>
__device__ __forceinline__ T mval(const uint8_t* m, int64_t k) {
  return m ? (m[k] ? T(1) : T(0)) : T(1);
}

__device__ __forceinline__ int lin_tid() {
  return threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
}

// Sums of NV values over the block into partials: block ``bid`` of ``nblk``
// stores value k at partials[k * nblk + bid].
template <int NV, int kThreads, typename A>
__device__ __forceinline__ void block_partials(const A (&v)[NV], double* partials, int64_t nblk,
                                               int64_t bid) {
  static_assert(NV <= 64, "one summing thread per value");
  __shared__ double red[kThreads / 64][NV];
  const int tid = lin_tid();
  const int lane = tid & 63, wid = tid >> 6;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const A s = wave_sum_last(v[k]);
    if (lane == 63) red[wid][k] = (double)s;
  }
  __syncthreads();
  if (tid < NV) {
    // Value-major: value k of block b at partials[k * nblocks + b], so the
    // finishing kernel's reads are coalesced.  One thread per value sums the
    // waves in order.
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w) s += red[w][tid];
    partials[tid * nblk + bid] = s;
  }
}
template <int NV, int kThreads, typename A>
__device__ __forceinline__ void block_partials(const A (&v)[NV], double* partials) {
  block_partials<NV, kThreads>(v, partials, (int64_t)gridDim.x * gridDim.y,
                               (int64_t)blockIdx.y * gridDim.x + blockIdx.x);
}

// Order of the PCG dots (z = M r, a = A z, q = q_{k-1} = A p_{k-1}).
enum CgDot : int { kZR, kZQ, kZA, kRR, kRA, kRQ, kAA, kAQ, kQQ, kNumCgDots };

// ---------------------------------------------------------------------------
// Tiled smoother kernel.  MODE:
//   0 SMOOTH   : NS sweeps                                  -> u_out
//   1 DOWN     : NS sweeps, residual, restriction           -> u_out, C.b
//   2 UP       : u += P(C.u), NS sweeps                     -> u_out
//   3 UP_CG    : as UP with one more halo ring, then a = A z on the tile
//                interior -> u_out (z), az_out (a), and the nine PCG dots of
//                z, a, r (= b) and q_{k-1} (= w)
//   4 DOWN_STEP: (wavefront tiles only) the previous PCG step on the tile,
//                then DOWN from zero on the new residual -> upd.q_out,
//                upd.r_out, upd.p, upd.x, u_out, C.b
// ---------------------------------------------------------------------------
enum TileMode : int { kSmooth = 0, kDown = 1, kUp = 2, kUpCG = 3, kDownUpd = 4 };

// The PCG step that the level-0 down kernel of the next V-cycle applies
// first (kDownUpd; wavefront tiles only): with a = A z,
// q_out = a + beta q_in, r_out = r_in - alpha q_out, p = z + beta p,
// x += alpha p.  r_in and q_in are read on the tile's halo as well, so they
// cannot be the arrays written.
template <typename T>
struct PcgUpdArgs {
  const T* z;
  T* p;
  T* x;
  int64_t ld_x;
  const T* q_in;
  T* q_out;
  const T* r_in;  // passed to the kernel as its b
  T* r_out;
};

constexpr int kTx = 64, kTy = 16, kTileThreads = 256;

template <typename T>
struct TileArgs {
  LevelDev<T> L, C;
  const T* u_in;
  const T* b;
  T* u_out;
  const T* w;
  T* az_out;
  T omw[3];  // the weight of sweep k (the plan's omega unless it smooths with
             // Chebyshev weights)
  double* partials;
  PcgScalars* sc;
  int tiles_x, ntiles;
  PcgUpdArgs<T> upd;  // kDownUpd; b is r_in
};

}  // namespace fvx
