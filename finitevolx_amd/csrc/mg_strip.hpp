// Strip kernels: damped-Jacobi sweeps with their transfers and PCG dots on
// one level, for every level the FP32 Dirichlet wave tiles (mg.hip) do not
// run (the no-flux operator with variable coefficients, and FP64).
#pragma once

#include "mg_level.hpp"

namespace fvx {

// Sweeps one launch can fuse (1, 2, 3 or 6).
constexpr int kStripMaxFuse = 6;

// Largest block count of a launch on an ny x nx level (partials of kUpCG).
inline int64_t strip_max_blocks(int ny, int nx) {
  return ((int64_t)cdiv(nx, 64 - 2 * (kStripMaxFuse + 1)) * cdiv(ny, 4) + 3) / 4;
}

// Run ``ns`` sweeps of mode ``mode`` (kSmooth, kDown, kUp, kUpCG) on a.L from
// a.u_in (from zero when ``zero``), sweep k weighted by a.omw[k % 3]; returns
// the number of blocks (kUpCG: each wrote its partial dots).
template <typename T, int KIND>
int launch_strip(int ns, int mode, bool zero, TileArgs<T> a, hipStream_t s);
extern template int launch_strip<double, kNoflux>(int, int, bool, TileArgs<double>, hipStream_t);
extern template int launch_strip<float, kNoflux>(int, int, bool, TileArgs<float>, hipStream_t);
extern template int launch_strip<double, kDirichlet>(int, int, bool, TileArgs<double>,
                                                     hipStream_t);

}  // namespace fvx
