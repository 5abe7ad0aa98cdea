// Kernel of mg_strip.hpp (instantiated per operator and precision by the
// mg_strip_*.hip files).
//
// One wavefront owns a strip of 64 columns (64 - 2H of them written) and
// ``len`` rows and marches north: lane i holds column i of everything.  When
// row y arrives, sweep s updates row y - s from the values sweep s - 1 left
// on rows y - s - 1 .. y - s + 1, so all NS sweeps (and the residual or A z
// one row behind the last) cost one pass over the level's arrays, and the
// rows in flight are a few registers per array: b, the face coefficients and
// the inverse diagonal of the last NS + 1 rows, two rows of each sweep's
// iterate and its last north flux (the next row's south flux).  East
// neighbours and west fluxes are DPP lane moves: no LDS, no barriers.  Rows
// arrive in chunks of four, the next chunk's loads issued before the current
// chunk is swept.
//
// Bound: at 2048^2 (FP64, no-flux) the ~6 arrays of 33.5 MB a pass moves (the up
// leg with the dots 71 us, 4.6 TB/s); below, the march itself: at 1024^2 with six
// sweeps 2.5 wavefronts a SIMD keep the VALU at 0.45 of its issue peak and the
// memory at 0.29 (28 us), from 512^2 down a launch is one wavefront's rows one
// after the other (8-16 us).  The LDS tiles this replaces spent their time on LDS
// traffic and barriers (10 LDS accesses a cell and sweep) with too few waves to
// hide either.
// Halo: rows cost (len + 2H) / len, columns 64 / (64 - 2H); strip_rows picks
// len, long strips where the level fills the chip with them.
#pragma once

#include "mg_strip.hpp"

namespace fvx {

// Value of lane + 1 / lane - 1 (0 in the wave's last / first lane).
template <typename T>
__device__ __forceinline__ T strip_east(T v) {
  return dpp_move<0x130>(v);
}
template <typename T>
__device__ __forceinline__ T strip_west(T v) {
  return dpp_move<0x138>(v);
}

// Bit t = the mask of row row0 + t (t = 0 .. 63) in column col, 0 outside the
// level; row0 may be negative.  mcol: the column-packed mask, null = all wet.
__device__ __forceinline__ uint64_t strip_bits(const uint32_t* __restrict__ mcol, int ny, int nx,
                                               int col, int row0) {
  if (!mcol) {
    const int lo = max(0, -row0), hi = min(64, ny - row0);
    if (hi <= lo) return 0;
    const uint64_t upto = hi >= 64 ? ~uint64_t(0) : (uint64_t(1) << hi) - 1;
    return upto & ~((uint64_t(1) << lo) - 1);
  }
  const int g = max(row0, 0), blk = g >> 5, last = ny / 32 + 1, off = g & 31;
  const uint64_t w0 = mcol[(int64_t)min(blk, last) * nx + col];
  const uint64_t w1 = mcol[(int64_t)min(blk + 1, last) * nx + col];
  const uint64_t w2 = mcol[(int64_t)min(blk + 2, last) * nx + col];
  uint64_t v = ((w1 << 32) | w0) >> off;
  if (off) v |= w2 << (64 - off);
  return v << (g - row0);
}

// Halo of a launch: one ring per stencil sweep (the first sweep from a zero
// guess reads no neighbours) and one for the residual / A z.
template <int NS, int MODE, bool ZERO>
constexpr int strip_halo() {
  return NS - (ZERO ? 1 : 0) + ((MODE == kDown || MODE == kUpCG) ? 1 : 0);
}

constexpr int kStripChunk = 4;

// BITS = false: an all-wet level whose strip, halo and coarse stencil lie
// inside it (no masks, no range checks).
template <typename T, int KIND, int NS, int MODE, bool ZERO, bool BITS>
__device__ __forceinline__ void strip_body(const TileArgs<T>& a, int i0, int j0, int j1, int lane,
                                           double (&dots)[kNumCgDots]) {
  constexpr int ST = NS - (ZERO ? 1 : 0);  // stencil sweeps
  constexpr bool RES = MODE == kDown || MODE == kUpCG;
  constexpr bool UP = MODE == kUp || MODE == kUpCG;
  constexpr bool NF = KIND == kNoflux;
  constexpr int H = strip_halo<NS, MODE, ZERO>();
  constexpr int L1 = ST + (RES ? 1 : 0);  // oldest row used by a stage: y - L1
  constexpr int CH = kStripChunk;
  constexpr int W = L1 + 1;  // rows y .. y - L1
  const LevelDev<T>& L = a.L;
  const int gi = i0 - H + lane;
  const bool colin = gi >= 0 && gi < L.nx;
  const bool lout = lane >= H && lane < 64 - H && gi < L.nx;
  const unsigned gic = (unsigned)min(max(gi, 0), L.nx - 1);
  const int y0 = j0 - H, nch = (j1 - j0 + 2 * H + CH - 1) / CH;

  // Mask bits of this lane's column from row y0 (wet and inside the level);
  // mh keeps the last rows' bits (bit s = row y - s).
  uint64_t mw = 0;
  uint32_t mh = 0;
  if constexpr (BITS) mw = colin ? strip_bits(L.mcol, L.ny, L.nx, (int)gic, y0) : 0;
  const bool edge = BITS && (y0 < 0 || y0 + nch * CH > L.ny || i0 - H < 0 || i0 - H + 64 > L.nx);

  // Coarse columns of the prolongation: I = gi / 2 and its neighbour In on
  // the side of gi; coarse rows from cr0, two per chunk.
  constexpr int K0 = (-H) >> 1;
  const int cr0 = (j0 >> 1) + K0 - 1;
  unsigned Ic = 0, Inc = 0;
  uint64_t cwI = 0, cwN = 0;
  if constexpr (UP) {
    const int I = gi >> 1, In = I + ((gi & 1) ? 1 : -1);
    Ic = (unsigned)min(max(I, 0), a.C.nx - 1);
    Inc = (unsigned)min(max(In, 0), a.C.nx - 1);
    if constexpr (BITS) {
      cwI = (I >= 0 && I < a.C.nx) ? strip_bits(a.C.mcol, a.C.ny, a.C.nx, (int)Ic, cr0) : 0;
      cwN = (In >= 0 && In < a.C.nx) ? strip_bits(a.C.mcol, a.C.ny, a.C.nx, (int)Inc, cr0) : 0;
    }
  }
  // Row-combined coarse values 3 v_I + v_In and weights 3 m_I + m_In of the
  // four coarse rows a chunk touches.
  T cw[UP ? 4 : 1];
  int cd[UP ? 4 : 1];
  T cnI[2], cnN[2];
  auto coarse_load = [&](int J, T& vI, T& vN) {
    const T* p = a.C.u + (int64_t)min(max(J, 0), a.C.ny - 1) * a.C.nx;
    vI = p[Ic];
    vN = p[Inc];
  };
  auto coarse_row = [&](T vI, T vN, T& w, int& d) {
    if constexpr (BITS) {
      const int mI = (int)(cwI & 1), mN = (int)(cwN & 1);
      cwI >>= 1;
      cwN >>= 1;
      w = T(3) * (mI ? vI : T(0)) + (mN ? vN : T(0));
      d = 3 * mI + mN;
    } else {
      w = T(3) * vI + vN;
      d = 4;
    }
  };

  // Next chunk's rows.
  T nb[CH], nu[ZERO ? 1 : CH], ncx[NF ? CH : 1], ncy[NF ? CH : 1], niv[NF ? CH : 1];
  T nq[MODE == kUpCG ? CH : 1];
  const bool first = MODE == kUpCG ? a.sc->first != 0 : false;
  auto load_chunk = [&](int c) {
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      const int y = y0 + c * CH + k;
      const int64_t ro = (int64_t)min(max(y, 0), L.ny - 1) * L.nx;
      nb[k] = (a.b + ro)[gic];
      if constexpr (!ZERO) nu[k] = (a.u_in + ro)[gic];
      if constexpr (NF) {
        ncx[k] = (L.cx + ro)[gic];
        ncy[k] = (L.cy + ro)[gic];
        niv[k] = (L.inv + ro)[gic];
      }
      if constexpr (MODE == kUpCG) {
        const int64_t rq = (int64_t)min(max(y - L1, 0), L.ny - 1) * L.nx;
        nq[k] = (a.w + rq)[gic];
      }
    }
    if constexpr (UP) {
#pragma unroll
      for (int p = 0; p < 2; ++p) coarse_load(cr0 + 2 * c + 2 + p, cnI[p], cnN[p]);
    }
  };
  if constexpr (UP) {
    T vI[2], vN[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) coarse_load(cr0 + p, vI[p], vN[p]);
    load_chunk(0);
#pragma unroll
    for (int p = 0; p < 2; ++p) coarse_row(vI[p], vN[p], cw[2 + p], cd[2 + p]);
  } else {
    load_chunk(0);
  }
  // (the flag's round trip overlaps the first loads)
  if (a.sc && a.sc->done) return;

  const T idx2 = L.idx2, idy2 = L.idy2, lam = L.lam;
  T wb[W], wx[NF ? W : 1], wy[NF ? W : 1], wi[NF ? W : 1];
  T U[L1 + 1], US[NF ? 1 : L1 + 1], F[NF ? L1 + 1 : 1];
#pragma unroll
  for (int k = 0; k < W; ++k) wb[k] = T(0);
#pragma unroll
  for (int k = 0; k < (NF ? W : 1); ++k) wx[k] = wy[k] = wi[k] = T(0);
#pragma unroll
  for (int k = 0; k <= L1; ++k) U[k] = T(0);
#pragma unroll
  for (int k = 0; k < (NF ? 1 : L1 + 1); ++k) US[k] = T(0);
#pragma unroll
  for (int k = 0; k < (NF ? L1 + 1 : 1); ++k) F[k] = T(0);
  T res0 = T(0);  // residual of the even row of a restriction pair
  T d[kNumCgDots];

  // A u on the row of stage s (row y - s; stage s's input is U[s - 1], its
  // north neighbour un), before the mask.
  auto apply = [&](int s, T un) -> T {
    const T c = U[s - 1];
    T lap;
    if constexpr (NF) {
      const T fe = wx[s] * (strip_east(c) - c);
      const T fw = strip_west(fe);
      const T fn = wy[s] * (un - c);
      lap = (fe - fw) * idx2 + (fn - F[s - 1]) * idy2;
      F[s - 1] = fn;
    } else {
      lap = (strip_east(c) + strip_west(c) - T(2) * c) * idx2 +
            (un + US[s - 1] - T(2) * c) * idy2;
    }
    return lap - lam * c;
  };

  for (int c = 0; c < nch; ++c) {
    T cb[CH], cu[ZERO ? 1 : CH], ccx[NF ? CH : 1], ccy[NF ? CH : 1], civ[NF ? CH : 1];
    T cq[MODE == kUpCG ? CH : 1];
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      cb[k] = nb[k];
      if constexpr (!ZERO) cu[k] = nu[k];
      if constexpr (NF) {
        ccx[k] = ncx[k];
        ccy[k] = ncy[k];
        civ[k] = niv[k];
      }
      if constexpr (MODE == kUpCG) cq[k] = nq[k];
    }
    if constexpr (UP) {
      cw[0] = cw[2];
      cw[1] = cw[3];
      cd[0] = cd[2];
      cd[1] = cd[3];
#pragma unroll
      for (int p = 0; p < 2; ++p) coarse_row(cnI[p], cnN[p], cw[2 + p], cd[2 + p]);
    }
    if (c + 1 < nch) load_chunk(c + 1);
    if constexpr (MODE == kUpCG) {
#pragma unroll
      for (int k = 0; k < kNumCgDots; ++k) d[k] = T(0);
    }
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      const int y = y0 + c * CH + k;
      if constexpr (BITS) {
        mh = (mh << 1) | (uint32_t)(mw & 1);
        mw >>= 1;
        if (edge) {  // cells outside the level: no fluxes, no update
          const bool in = colin && y >= 0 && y < L.ny;
          cb[k] = in ? cb[k] : T(0);
          if constexpr (NF) {
            ccx[k] = in ? ccx[k] : T(0);
            ccy[k] = in ? ccy[k] : T(0);
            civ[k] = in ? civ[k] : T(0);
          }
        }
      }
      auto wet = [&](int s) -> T { return BITS ? (((mh >> s) & 1u) ? T(1) : T(0)) : T(1); };
#pragma unroll
      for (int q = W - 1; q > 0; --q) {
        wb[q] = wb[q - 1];
        if constexpr (NF) {
          wx[q] = wx[q - 1];
          wy[q] = wy[q - 1];
          wi[q] = wi[q - 1];
        }
      }
      wb[0] = cb[k];
      if constexpr (NF) {
        wx[0] = ccx[k];
        wy[0] = ccy[k];
        wi[0] = civ[k];
      }
      // Row y of the first iterate.
      T nw;
      if constexpr (ZERO) {
        if constexpr (NF) nw = a.omw[0] * wi[0] * wb[0];
        else nw = a.omw[0] * L.inv_d * wb[0];
        if constexpr (BITS && !NF) nw = nw * wet(0);
      } else {
        nw = cu[k];
        if constexpr (BITS) nw = nw * wet(0);  // u * mask (multigrid.py:383)
        if constexpr (UP) {
          // u = (u + P e_c) * mask (multigrid.py:875-876), _prolongate
          // (:510-603): row weights 3 / 1 of the coarse row and the one on
          // the side of y, normalised by the wet weights (no-flux).
          const int p = ((k - H) >> 1) - K0 + 1, pn = p + (((k - H) & 1) ? 1 : -1);
          const T w = T(3) * cw[p] + cw[pn];
          T e = w * T(0.0625);
          if constexpr (NF && BITS) {
            const int dd = 3 * cd[p] + cd[pn];
            if (__ballot(dd != 16) != 0) e = dd == 16 ? e : w / (T)max(dd, 1);
          }
          nw = nw + e;
          if constexpr (BITS) nw = nw * wet(0);
        }
      }
#pragma unroll
      for (int s = 1; s <= ST; ++s) {
        const T om = a.omw[(s - 1 + (ZERO ? 1 : 0)) % 3];
        const T un = nw;
        const T cc = U[s - 1];
        const T au = apply(s, un);
        T inv;
        if constexpr (NF) inv = wi[s];
        else inv = L.inv_d;
        nw = cc + om * inv * (wb[s] - au);
        if constexpr (BITS && !NF) nw = nw * wet(s);
        if constexpr (!NF) US[s - 1] = cc;
        U[s - 1] = un;
      }
      // nw: the last sweep's row y - ST.
      if constexpr (MODE != kUpCG) {
        const int r = y - ST;
        if (r >= j0 && r < j1 && lout) (a.u_out + (int64_t)r * L.nx)[gi] = nw;
      }
      if constexpr (RES) {
        const int r = y - L1;
        const T z = U[L1 - 1];
        T au = apply(L1, nw);
        if constexpr (!NF) US[L1 - 1] = z;
        U[L1 - 1] = nw;
        if constexpr (MODE == kDown) {
          // r = (b - A u) m; 2x2 restriction (multigrid.py:464-507; the
          // Dirichlet hierarchy's sum / 4): an odd row closes the pair, the
          // column pair through one lane move.  j0 is even and H = L1, so
          // row r is odd where k is.
          T rs = wb[L1] - au;
          if constexpr (BITS) rs = rs * wet(L1);
          if (k & 1) {
            const T s2 = res0 + rs;
            const T s4 = s2 + strip_east(s2);
            T f = T(0.25);
            if constexpr (BITS) {
              const int c2 = (int)((mh >> L1) & 1u) + (int)((mh >> (L1 + 1)) & 1u);
              const int c4 = c2 + __builtin_amdgcn_mov_dpp(c2, 0x130, 0xf, 0xf, true);
              if constexpr (NF)
                f = c4 == 4 ? T(0.25) : c4 == 3 ? T(1) / T(3) : c4 == 2 ? T(0.5) : T(1);
              // a coarse cell is wet with two or more wet children
              if (c4 < 2) f = T(0);
            }
            if (r >= j0 && r < j1 && lout && !(gi & 1))
              (a.C.b + (int64_t)(r >> 1) * a.C.nx)[gi >> 1] = s4 * f;
          } else {
            res0 = rs;
          }
        } else {
          if (r >= j0 && r < j1) {
            if constexpr (BITS) au = au * wet(L1);
            const T az = lout ? au : T(0), rd = lout ? wb[L1] : T(0);
            const T qd = (lout && !first) ? cq[k] : T(0);
            d[kZR] += z * rd;
            d[kZQ] += z * qd;
            d[kZA] += z * az;
            d[kRR] += rd * rd;
            d[kRA] += rd * az;
            d[kRQ] += rd * qd;
            d[kAA] += az * az;
            d[kAQ] += az * qd;
            d[kQQ] += qd * qd;
            if (lout) {
              (a.u_out + (int64_t)r * L.nx)[gi] = z;
              (a.az_out + (int64_t)r * L.nx)[gi] = az;
            }
          }
        }
      }
    }
    if constexpr (MODE == kUpCG) {
#pragma unroll
      for (int k = 0; k < kNumCgDots; ++k) dots[k] += (double)d[k];
    }
  }
}

template <typename T, int KIND, int NS, int MODE, bool ZERO>
__global__ __launch_bounds__(256) void mg_strip_kernel(TileArgs<T> a, int len) {
  constexpr int H = strip_halo<NS, MODE, ZERO>();
  const int lane = threadIdx.x & 63;
  const int bx = xcd_swizzle(blockIdx.x, gridDim.x);
  // (scalar, so that every per-strip quantity and branch is uniform)
  const int tile = __builtin_amdgcn_readfirstlane(bx * 4 + (threadIdx.x >> 6));
  double dots[kNumCgDots];
#pragma unroll
  for (int k = 0; k < kNumCgDots; ++k) dots[k] = 0.0;
  if (tile < a.ntiles) {
    const int ty = tile / a.tiles_x;
    const int i0 = (tile - ty * a.tiles_x) * (64 - 2 * H);
    const int j0 = ty * len, j1 = min(j0 + len, a.L.ny);
    // (two more cells cover the prolongation stencil, chunk - 1 rows more the
    // last chunk's rows)
    const bool inner = !a.L.mcol && !a.C.mcol && j0 - H - 2 >= 0 && i0 - H - 2 >= 0 &&
                       j0 + len + H + kStripChunk + 1 < a.L.ny && i0 - H + 66 < a.L.nx;
    if (inner) strip_body<T, KIND, NS, MODE, ZERO, false>(a, i0, j0, j1, lane, dots);
    else strip_body<T, KIND, NS, MODE, ZERO, true>(a, i0, j0, j1, lane, dots);
  }
  if constexpr (MODE == kUpCG) {
    if (a.sc->done) return;
    block_partials<kNumCgDots, 256>(dots, a.partials, gridDim.x, bx);
  }
}

// Rows per strip: as many as leave two wavefronts per SIMD (2048), at most 32
// (the mask windows hold 64 rows with the halo), at least 4.  Short strips sweep
// more halo rows than they keep, and are still the fastest where long ones would
// leave SIMDs empty: us of a V-cycle with 3 (6) sweeps a leg, no-flux FP64, by
// this rule / all levels with 4, 8, 16, 32 rows:
//   256^2      52 (74)   / 52 (74)   58 (81)   70 (95)   92 (123)
//   512^2      70 (101)  / 70 (101)  75 (105)  93 (127) 128 (169)
//   1024^2    105 (149)  / 109 (161) 109 (153) 126 (171) 166 (217)
//   600x1000   68 (155)  / 68 (155)  74 (169)  92 (205) 137 (295)
//   2048^2    192 (253)  / 226 (370) 199 (292) 212 (278) 255 (319)
// (FP32 and the Dirichlet operator likewise.)
inline int strip_rows(int tiles_x, int ny) {
  int len = 32;
  while (len > 4 && (int64_t)tiles_x * cdiv(ny, len) < 2048) len /= 2;
  return len;
}

template <typename T, int KIND, int NS, int MODE, bool ZERO>
static int strip_go(TileArgs<T>& a, hipStream_t s) {
  constexpr int H = strip_halo<NS, MODE, ZERO>();
  a.tiles_x = cdiv(a.L.nx, 64 - 2 * H);
  const int len = strip_rows(a.tiles_x, a.L.ny);
  a.ntiles = a.tiles_x * cdiv(a.L.ny, len);
  const int nblk = cdiv(a.ntiles, 4);
  hipLaunchKernelGGL((mg_strip_kernel<T, KIND, NS, MODE, ZERO>), dim3(nblk), dim3(256), 0, s, a,
                     len);
  return nblk;
}

template <typename T, int KIND, int NS>
static int strip_mode(int mode, bool zero, TileArgs<T>& a, hipStream_t s) {
  switch (mode) {
    case kSmooth:
      return zero ? strip_go<T, KIND, NS, kSmooth, true>(a, s)
                  : strip_go<T, KIND, NS, kSmooth, false>(a, s);
    case kDown:
      return zero ? strip_go<T, KIND, NS, kDown, true>(a, s)
                  : strip_go<T, KIND, NS, kDown, false>(a, s);
    case kUp:
      return strip_go<T, KIND, NS, kUp, false>(a, s);
    default:
      return strip_go<T, KIND, NS, kUpCG, false>(a, s);
  }
}

template <typename T, int KIND>
int launch_strip(int ns, int mode, bool zero, TileArgs<T> a, hipStream_t s) {
  switch (ns) {
    case 1: return strip_mode<T, KIND, 1>(mode, zero, a, s);
    case 2: return strip_mode<T, KIND, 2>(mode, zero, a, s);
    case 3: return strip_mode<T, KIND, 3>(mode, zero, a, s);
    default: return strip_mode<T, KIND, 6>(mode, zero, a, s);
  }
}

}  // namespace fvx
