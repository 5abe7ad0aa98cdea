#include "mg_coarse.hpp"

namespace fvx {

constexpr int kCoarseThreads = 1024;

// LDS-resident coarse V-cycle of a hierarchy whose level lc is larger than
// kCoarseCells (batched members whose grid stops halving early).  Levels
// lc .. nl-1 keep their iterate u, scratch t and right-hand side b in dynamic
// LDS, addressed by cell offsets (ds_read/ds_write); the 1024 threads tile
// each level as 32 x 32 blocks of cells, so no integer division is needed.  Every stored iterate is already
// multiplied by its mask, which is the reference's u * mask before the
// stencil (multigrid.py:383).
template <typename T, int KIND>
struct CoarseLds {
  T* sm;
  __device__ __forceinline__ T m_at(const LevelDev<T>& L, int k) const {
    return mval<T>(L.mask, k);
  }
  __device__ __forceinline__ T inv_at(const LevelDev<T>& L, int k, T m) const {
    if constexpr (KIND == kDirichlet) return L.inv_d * m;
    return L.inv[k];
  }
  // (A u)(j, i) for u at LDS offset ou (zero outside the level).
  __device__ __forceinline__ T Au(const LevelDev<T>& L, int ou, int j, int i, int k, T m) const {
    const T c = sm[ou + k];
    const T e = (i + 1 < L.nx) ? sm[ou + k + 1] : T(0);
    const T w = (i > 0) ? sm[ou + k - 1] : T(0);
    const T n = (j + 1 < L.ny) ? sm[ou + k + L.nx] : T(0);
    const T s = (j > 0) ? sm[ou + k - L.nx] : T(0);
    T lap;
    if constexpr (KIND == kDirichlet) {
      lap = (e + w - T(2) * c) * L.idx2 + (n + s - T(2) * c) * L.idy2;
    } else {
      const T cxe = L.cx[k], cxw = (i > 0) ? L.cx[k - 1] : T(0);
      const T cyn = L.cy[k], cys = (j > 0) ? L.cy[k - L.nx] : T(0);
      lap = (cxe * (e - c) - cxw * (c - w)) * L.idx2 + (cyn * (n - c) - cys * (c - s)) * L.idy2;
    }
    return (lap - L.lam * c) * m;
  }
  // n damped-Jacobi sweeps of level L (u at ou, scratch at ot, b at ob); the
  // result ends in ou.
  __device__ void sweeps(const LevelDev<T>& L, int ou, int ot, int ob, int n, bool zero,
                         const T* w, int tx, int ty) const {
    int src = ou, dst = ot;
    for (int sw = 0; sw < n; ++sw) {
      const T om = w[sw < kMaxW ? sw : kMaxW - 1];
      for (int j = ty; j < L.ny; j += 32)
        for (int i = tx; i < L.nx; i += 32) {
          const int k = j * L.nx + i;
          const T m = m_at(L, k);
          const T inv = inv_at(L, k, m);
          T un;
          if (zero && sw == 0) un = (om * inv * sm[ob + k]) * m;
          else un = (sm[src + k] + om * inv * (sm[ob + k] - Au(L, src, j, i, k, m))) * m;
          sm[dst + k] = un;
        }
      __syncthreads();
      const int tmp = src;
      src = dst;
      dst = tmp;
    }
    if (src != ou) {  // odd number of sweeps: copy back
      for (int j = ty; j < L.ny; j += 32)
        for (int i = tx; i < L.nx; i += 32) sm[ou + j * L.nx + i] = sm[src + j * L.nx + i];
      __syncthreads();
    }
  }
};

template <typename T, int KIND>
__device__ __forceinline__ void mg_coarse_large_body(const CoarseArgs<T>& a,
                                                     unsigned char* coarse_smem,
                                                     int (*tab)[16]) {
  const bool skip = a.done && *a.done;
  CoarseLds<T, KIND> S{reinterpret_cast<T*>(coarse_smem)};
  T* sm = S.sm;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  // LDS offsets of each level's u, t, b (a table in LDS: indexed by the
  // runtime level, a private array would live in scratch memory).
  int *ou = tab[0], *ot = tab[1], *ob = tab[2];
  if (threadIdx.x == 0) {
    int o = 0;
    for (int l = a.lc; l < a.nl; ++l) {
      const int n = a.lv[l].ny * a.lv[l].nx;
      ou[l] = o;
      ot[l] = o + n;
      ob[l] = o + 2 * n;
      o += 3 * n;
    }
  }
  __syncthreads();
  // Level lc's right-hand side (and masked guess) from global memory.
  {
    const LevelDev<T>& G = a.lv[a.lc];
    for (int j = ty; j < G.ny; j += 32)
      for (int i = tx; i < G.nx; i += 32) {
        const int k = j * G.nx + i;
        sm[ob[a.lc] + k] = G.b[k];
        if (a.nonzero_init) sm[ou[a.lc] + k] = G.u[k] * S.m_at(G, k);
      }
    if (skip) return;
    __syncthreads();
  }
  // Down leg: pre-smoothing, residual, mask-weighted 2x2 restriction.
  for (int l = a.lc; l < a.nl - 1; ++l) {
    const LevelDev<T>& L = a.lv[l];
    const LevelDev<T>& C = a.lv[l + 1];
    const bool zero = !(a.nonzero_init && l == a.lc);
    if (a.n_pre > 0) {
      S.sweeps(L, ou[l], ot[l], ob[l], a.n_pre, zero, a.w[0], tx, ty);
    } else if (zero) {
      for (int j = ty; j < L.ny; j += 32)
        for (int i = tx; i < L.nx; i += 32) sm[ou[l] + j * L.nx + i] = T(0);
      __syncthreads();
    }
    // residual r = (b - A u) m into the scratch array
    for (int j = ty; j < L.ny; j += 32)
      for (int i = tx; i < L.nx; i += 32) {
        const int k = j * L.nx + i;
        const T m = S.m_at(L, k);
        sm[ot[l] + k] = (sm[ob[l] + k] - S.Au(L, ou[l], j, i, k, m)) * m;
      }
    __syncthreads();
    for (int J = ty; J < C.ny; J += 32)
      for (int I = tx; I < C.nx; I += 32) {
        const int f = (2 * J) * L.nx + 2 * I;
        const T m00 = S.m_at(L, f), m01 = S.m_at(L, f + 1), m10 = S.m_at(L, f + L.nx),
                m11 = S.m_at(L, f + L.nx + 1);
        const T s4 = sm[ot[l] + f] * m00 + sm[ot[l] + f + 1] * m01 + sm[ot[l] + f + L.nx] * m10 +
                     sm[ot[l] + f + L.nx + 1] * m11;
        const T cnt = m00 + m01 + m10 + m11;
        const int kc = J * C.nx + I;
        const T rs = KIND == kDirichlet ? s4 * T(0.25) : s4 / (cnt > T(1) ? cnt : T(1));
        sm[ob[l + 1] + kc] = rs * S.m_at(C, kc);
      }
    __syncthreads();
  }
  // Bottom solve.
  {
    const int lb = a.nl - 1;
    const LevelDev<T>& B = a.lv[lb];
    const bool zero = !(a.nonzero_init && a.lc == lb);
    if (a.n_coarse > 0) {
      S.sweeps(B, ou[lb], ot[lb], ob[lb], a.n_coarse, zero, a.w[2], tx, ty);
    } else if (zero) {
      for (int j = ty; j < B.ny; j += 32)
        for (int i = tx; i < B.nx; i += 32) sm[ou[lb] + j * B.nx + i] = T(0);
      __syncthreads();
    }
  }
  // Up leg: u += P(u_c) (9/3/3/1 weights, mask renormalised), post-smoothing.
  for (int l = a.nl - 2; l >= a.lc; --l) {
    const LevelDev<T>& L = a.lv[l];
    const LevelDev<T>& C = a.lv[l + 1];
    for (int j = ty; j < L.ny; j += 32)
      for (int i = tx; i < L.nx; i += 32) {
        const int k = j * L.nx + i;
        const T m = S.m_at(L, k);
        const int J = j >> 1, I = i >> 1;
        const int sj = (j & 1) ? 1 : -1, si = (i & 1) ? 1 : -1;
        auto vm = [&](int jj, int ii, T& mm) -> T {
          if (jj < 0 || jj >= C.ny || ii < 0 || ii >= C.nx) {
            mm = T(0);
            return T(0);
          }
          const int kc = jj * C.nx + ii;
          mm = S.m_at(C, kc);
          return sm[ou[l + 1] + kc];  // stored iterates are already masked
        };
        T mc, mx, my, md;
        const T vc = vm(J, I, mc), vx = vm(J, I + si, mx), vy = vm(J + sj, I, my),
                vd = vm(J + sj, I + si, md);
        const T w = T(9) * vc + T(3) * vx + T(3) * vy + vd;
        const T d = T(9) * mc + T(3) * mx + T(3) * my + md;
        const T e = KIND == kDirichlet ? w * T(0.0625) : w / (d > T(1) ? d : T(1));
        sm[ou[l] + k] = (sm[ou[l] + k] + e * m) * m;
      }
    __syncthreads();
    S.sweeps(L, ou[l], ot[l], ob[l], a.n_post, false, a.w[1], tx, ty);
  }
  // Level lc's corrected iterate back to global memory.
  {
    const LevelDev<T>& G = a.lv[a.lc];
    for (int j = ty; j < G.ny; j += 32)
      for (int i = tx; i < G.nx; i += 32) G.u[j * G.nx + i] = sm[ou[a.lc] + j * G.nx + i];
  }
}

// ---------------------------------------------------------------------------
// Coarse V-cycle of levels with at most kCoarseCells cells each.
//
// Everything a cycle reads is fetched in one go at the start: thread t keeps
// cells t, t + 1024, ... of level lc (Q of them: coefficients, right-hand
// side, iterate) in registers for the whole cycle, and the coarser levels
// (Q = 1) keep theirs in LDS, one flat array per quantity.  A sweep is four
// LDS reads and one write a cell and one barrier (two iterate buffers: the
// level's own and a scratch shared by all levels); a level of one wavefront's
// cells (the bottom, where most sweeps run) is swept by one wavefront without
// barriers.  A neighbour outside the level is a zero cell behind either
// buffer (no-flux: any cell, its face coefficient is zero).  Q is the
// kernel's, not the level's, so that the code a launch runs stays short: at
// this length its instructions are fetched once and used once or twice.
// Bound: one CU's VALU at 4096 cells (~20 operations a cell and sweep), the
// LDS round trip and barrier below.  Measured (64^2 down to 8^2, FP64 no-flux,
// 6 + 6 and 50 sweeps): 34 us, 107 us with every coefficient, mask and index
// division repeated in each sweep; FP32 Dirichlet, 3 + 3 and 4: 16 us, 36 us.
// ---------------------------------------------------------------------------

// k / n for 0 <= k < 4096 + 1024, 1 <= n <= 4096 (the quotient is at least
// 0.5 / n from an integer, the product's error below 2e-3 / n).
__device__ __forceinline__ int small_div(int k, float rn) { return (int)(((float)k + 0.5f) * rn); }

template <typename T, int KIND, int Q>
struct CoarseRegs {
  static constexpr bool NF = KIND == kNoflux;
  // A thread's cells of one level.
  template <int C>
  struct Cells {
    T inv[C], b[C], c[C];
    int wet;  // bit q: cell q is wet
    T xe[NF ? C : 1], xw[NF ? C : 1], yn[NF ? C : 1], ys[NF ? C : 1];
    int e[NF ? 1 : C], w[NF ? 1 : C], n[NF ? 1 : C], s[NF ? 1 : C];  // neighbour cells
    __device__ __forceinline__ T m(int q) const { return (wet >> q) & 1 ? T(1) : T(0); }
  };
  struct Geo {  // one level
    int ny, nx, N;
    T idx2, idy2;
    T* u;               // LDS: its iterate (N + 1 cells)
    const uint8_t* wm;  // LDS: its wet mask
  };
  T* ot;  // LDS: the scratch
  T lam;
  bool masked;

  template <int C>
  __device__ __forceinline__ void neighbours(const Geo& g, Cells<C>& r, int q, int kc, int j,
                                             int i) const {
    if constexpr (!NF) {
      r.e[q] = i + 1 < g.nx ? kc + 1 : g.N;
      r.w[q] = i > 0 ? kc - 1 : g.N;
      r.n[q] = j + 1 < g.ny ? kc + g.nx : g.N;
      r.s[q] = j > 0 ? kc - g.nx : g.N;
    }
  }
  // b - A u at cell q, u in the buffer ``u`` (dry cells: A u is zero, as their
  // iterate and every face coefficient are).
  template <int C>
  __device__ __forceinline__ T defect(const Geo& g, const Cells<C>& r, int q, const T* u) const {
    const T c = r.c[q];
    if constexpr (NF) {
      const int k = min((int)threadIdx.x + q * kCoarseThreads, g.N - 1);
      const T e = u[k + 1], w = u[max(k - 1, 0)], n = u[min(k + g.nx, g.N)],
              s = u[max(k - g.nx, 0)];
      const T lap = (r.xe[q] * (e - c) - r.xw[q] * (c - w)) * g.idx2 +
                    (r.yn[q] * (n - c) - r.ys[q] * (c - s)) * g.idy2;
      return r.b[q] - (lap - lam * c);
    } else {
      const T lap = (u[r.e[q]] + u[r.w[q]] - T(2) * c) * g.idx2 +
                    (u[r.n[q]] + u[r.s[q]] - T(2) * c) * g.idy2;
      return r.b[q] - (lap - lam * c) * r.m(q);
    }
  }
  // n sweeps from the iterate in r.c, which the caller has not stored
  // (``zero``: from zero, r.c unset): it is written to the buffer from which
  // the last sweep ends in g.u.
  template <int C, bool SOLO>
  __device__ __forceinline__ void sweep(const Geo& g, int n, bool zero, const T* wt,
                                        Cells<C>& r) const {
    T* dst = (n & 1) ? ot : g.u;
    auto sync = [&]() {
      if constexpr (SOLO) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      else __syncthreads();
    };
    auto put = [&]() {
#pragma unroll
      for (int q = 0; q < C; ++q) {
        const int k = threadIdx.x + q * kCoarseThreads;
        if (k < g.N) dst[k] = r.c[q];
      }
    };
    if (!SOLO || threadIdx.x < 64) {
      if (threadIdx.x == 0) g.u[g.N] = ot[g.N] = T(0);
      if (!zero || n == 0) {
        if (zero) {
#pragma unroll
          for (int q = 0; q < C; ++q) r.c[q] = T(0);
        }
        put();
      }
      sync();
      T om = wt[0];
      for (int s = 0; s < n; ++s) {
        const T next = wt[min(s + 1, kMaxW - 1)];
        const T* src = dst;
        dst = dst == ot ? g.u : ot;
        if (zero && s == 0) {
#pragma unroll
          for (int q = 0; q < C; ++q) r.c[q] = om * r.inv[q] * r.b[q];
        } else {
#pragma unroll
          for (int q = 0; q < C; ++q) r.c[q] = r.c[q] + om * r.inv[q] * defect(g, r, q, src);
        }
        put();
        sync();
        om = next;
      }
    }
    if constexpr (SOLO) __syncthreads();
  }
  __device__ __forceinline__ void sweeps(const Geo& g, int n, bool zero, const T* wt,
                                         Cells<1>& r) const {
    if (g.N <= 64) sweep<1, true>(g, n, zero, wt, r);
    else sweep<1, false>(g, n, zero, wt, r);
  }
  // The residual of g's iterate, restricted into cb (coarse level h).
  template <int C>
  __device__ __forceinline__ void restrict_to(const Geo& g, const Cells<C>& r, const Geo& h,
                                              T* cb) const {
#pragma unroll
    for (int q = 0; q < C; ++q) {
      const int k = threadIdx.x + q * kCoarseThreads;
      if (k < g.N) ot[k] = defect(g, r, q, g.u) * r.m(q);
    }
    __syncthreads();
    const int kc = threadIdx.x;
    if (kc < h.N) {
      const int J = small_div(kc, 1.0f / h.nx), I = kc - J * h.nx, f = 2 * J * g.nx + 2 * I;
      const T s4 = ot[f] + ot[f + 1] + ot[f + g.nx] + ot[f + g.nx + 1];
      T rs = s4 * T(0.25);
      if (masked) {
        const int cnt = g.wm[f] + g.wm[f + 1] + g.wm[f + g.nx] + g.wm[f + g.nx + 1];
        if (NF) rs = s4 / (T)max(cnt, 1);
        if (!h.wm[kc]) rs = T(0);
      }
      cb[kc] = rs;
    }
    __syncthreads();
  }
  // r.c = (u + P u_c) * mask (9/3/3/1 weights; no-flux: renormalised by the
  // wet ones), u the thread's cells of g's iterate, u_c the coarse level h's.
  template <int C>
  __device__ __forceinline__ void prolong(const Geo& g, const Geo& h, Cells<C>& r) const {
    const float rn = 1.0f / g.nx;
#pragma unroll
    for (int q = 0; q < C; ++q) {
      const int k = min((int)threadIdx.x + q * kCoarseThreads, g.N - 1);
      const int j = small_div(k, rn), i = k - j * g.nx;
      const int J = j >> 1, I = i >> 1;
      const int Jn = J + ((j & 1) ? 1 : -1), In = I + ((i & 1) ? 1 : -1);
      const bool inJ = Jn >= 0 && Jn < h.ny, inI = In >= 0 && In < h.nx;
      // (outside the level: the zero cell; stored iterates are masked)
      const int c0 = J * h.nx + I, cx = inI ? J * h.nx + In : h.N, cy = inJ ? Jn * h.nx + I : h.N,
                cd = inI && inJ ? Jn * h.nx + In : h.N;
      const T w = T(9) * h.u[c0] + T(3) * h.u[cx] + T(3) * h.u[cy] + h.u[cd];
      T e = w * T(0.0625);
      if constexpr (NF) {
        int d = 9 * h.wm[c0] + (inI ? 3 * h.wm[cx] : 0) + (inJ ? 3 * h.wm[cy] : 0) +
                (inI && inJ ? h.wm[cd] : 0);
        if (d != 16) e = w / (T)max(d, 1);
      }
      r.c[q] = (g.u[k] + e * r.m(q)) * r.m(q);
    }
  }
};

template <typename T, int KIND, int Q>
__device__ __forceinline__ void mg_coarse_lds_body(const CoarseArgs<T>& a,
                                                   unsigned char* coarse_smem) {
  using S_ = CoarseRegs<T, KIND, Q>;
  using Geo = typename S_::Geo;
  constexpr bool NF = S_::NF;
  const LevelDev<T>& L = a.lv[a.lc];
  const int tid = threadIdx.x, nd = a.nl - a.lc;
  const int ny = L.ny, nx = L.nx, N = ny * nx;
  const bool skip = a.done && *a.done;
  // Cells of the levels below lc (each a quarter of the one above).
  int low = 0;
  for (int d = 1; d < nd; ++d) low += (ny >> d) * (nx >> d);
  // LDS: scratch, u of level lc, then flat over the lower levels u (a zero
  // cell after each), b and (no-flux) cx, cy, 1 / diag per cell or (Dirichlet)
  // 1 / diag per level; wet masks as bytes.
  T* sm = reinterpret_cast<T*>(coarse_smem);
  T *fu = sm + 2 * (N + 1), *fb = fu + low + nd, *fx = fb + low, *fy = fx + low,
    *fi = NF ? fy + low : fx;
  uint8_t* wm = reinterpret_cast<uint8_t*>(NF ? fi + low : fi + nd);
  S_ S{sm, L.lam, L.mask != nullptr};
  Geo g0{ny, nx, N, L.idx2, L.idy2, sm + N + 1, wm};
  auto lower = [&](int d, int off) {  // level lc + d, its flat offset
    return Geo{ny >> d,
               nx >> d,
               (ny >> d) * (nx >> d),
               (T)ldexp(L.idx2, -2 * d),
               (T)ldexp(L.idy2, -2 * d),
               fu + off + d - 1,
               wm + N + off};
  };

  // Every load of the cycle: level lc's cells into registers ...
  typename S_::template Cells<Q> top;
  top.wet = 0;
  const float rn = 1.0f / nx;
  uint8_t m0[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int kc = min(tid + q * kCoarseThreads, N - 1);
    const int j = small_div(kc, rn), i = kc - j * nx;
    top.b[q] = L.b[kc];
    m0[q] = S.masked ? L.mask[kc] : 1;
    if (a.nonzero_init) top.c[q] = L.u[kc];
    if constexpr (NF) {
      top.inv[q] = L.inv[kc];
      top.xe[q] = L.cx[kc];
      top.xw[q] = i > 0 ? L.cx[kc - 1] : T(0);
      top.yn[q] = L.cy[kc];
      top.ys[q] = j > 0 ? L.cy[kc - nx] : T(0);
    }
    S.neighbours(g0, top, q, kc, j, i);
  }
  // ... and the lower levels' coefficients and masks, flat, into LDS.
  if constexpr (!NF) {
    if (tid < nd) fi[tid] = a.lv[a.lc + tid].inv_d;
  }
  if (low > 0 && (NF || S.masked)) {
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const int t = tid + p * kCoarseThreads;
      if (t >= low) break;
      int l = a.lc, k = 0;
      for (int d = 1, off = 0; d < nd; ++d) {
        const int n = (ny >> d) * (nx >> d);
        if (t >= off && t < off + n) {
          l = a.lc + d;
          k = t - off;
        }
        off += n;
      }
      const LevelDev<T>& B = a.lv[l];
      if constexpr (NF) {
        fx[t] = B.cx[k];
        fy[t] = B.cy[k];
        fi[t] = B.inv[k];
      }
      wm[N + t] = B.mask ? B.mask[k] : 1;
    }
  }
  if (skip) return;
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int k = tid + q * kCoarseThreads;
    if (k < N && (NF || S.masked)) wm[k] = m0[q];
    top.wet |= m0[q] ? 1 << q : 0;
    if constexpr (!NF) top.inv[q] = L.inv_d * (m0[q] ? T(1) : T(0));
    if (a.nonzero_init) top.c[q] = top.c[q] * (m0[q] ? T(1) : T(0));
  }
  __syncthreads();

  // A cell of level lc + d of this thread, from LDS.
  auto cell = [&](const Geo& g, int d, int off, typename S_::template Cells<1>& r) {
    const int kc = min(tid, g.N - 1), j = small_div(kc, 1.0f / g.nx), i = kc - j * g.nx;
    r.b[0] = fb[off + kc];
    r.wet = S.masked ? g.wm[kc] != 0 : 1;
    if constexpr (NF) {
      r.inv[0] = fi[off + kc];
      r.xe[0] = fx[off + kc];
      r.xw[0] = i > 0 ? fx[off + kc - 1] : T(0);
      r.yn[0] = fy[off + kc];
      r.ys[0] = j > 0 ? fy[off + kc - g.nx] : T(0);
    } else {
      // (the scalar of an all-wet level)
      r.inv[0] = r.wet ? fi[d] : T(0);
    }
    S.neighbours(g, r, 0, kc, j, i);
  };
  const bool zero0 = !a.nonzero_init;
  if (nd == 1) {
    S.template sweep<Q, false>(g0, a.n_coarse, zero0, a.w[2], top);
  } else {
    S.template sweep<Q, false>(g0, a.n_pre, zero0, a.w[0], top);
    S.restrict_to(g0, top, lower(1, 0), fb);
    int off = 0;
    typename S_::template Cells<1> r;
    for (int d = 1; d < nd; ++d) {
      const Geo g = lower(d, off);
      const bool last = d == nd - 1;
      cell(g, d, off, r);
      S.sweeps(g, last ? a.n_coarse : a.n_pre, true, last ? a.w[2] : a.w[0], r);
      if (!last) {
        S.restrict_to(g, r, lower(d + 1, off + g.N), fb + off + g.N);
        off += g.N;
      }
    }
    for (int d = nd - 2; d >= 1; --d) {
      const Geo h = lower(d + 1, off);
      off -= (ny >> d) * (nx >> d);
      const Geo g = lower(d, off);
      cell(g, d, off, r);
      S.prolong(g, h, r);
      S.sweeps(g, a.n_post, false, a.w[1], r);
    }
    S.prolong(g0, lower(1, 0), top);
    S.template sweep<Q, false>(g0, a.n_post, false, a.w[1], top);
  }
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int k = tid + q * kCoarseThreads;
    if (k < N) L.u[k] = top.c[q];
  }
}

template <typename T, int KIND, int Q>
__global__ __launch_bounds__(kCoarseThreads) void mg_coarse_lds_kernel(CoarseArgs<T> a) {
  extern __shared__ __align__(16) unsigned char coarse_smem[];
  mg_coarse_lds_body<T, KIND, Q>(a, coarse_smem);
}
// (a member whose level lc is small runs the batch's Q with its upper cells
// dead)
template <typename T, int KIND, int Q>
__global__ __launch_bounds__(kCoarseThreads) void mg_coarse_batch_kernel(
    const CoarseArgs<T>* __restrict__ args) {
  extern __shared__ __align__(16) unsigned char coarse_smem[];
  mg_coarse_lds_body<T, KIND, Q>(args[blockIdx.x], coarse_smem);
}
template <typename T, int KIND>
__global__ __launch_bounds__(kCoarseThreads) void mg_coarse_large_batch_kernel(
    const CoarseArgs<T>* __restrict__ args) {
  extern __shared__ __align__(16) unsigned char coarse_smem[];
  __shared__ int tab[3][16];
  mg_coarse_large_body<T, KIND>(args[blockIdx.x], coarse_smem, tab);
}

template <typename T>
size_t coarse_lds_bytes(const CoarseArgs<T>& a, bool large) {
  const size_t top = (size_t)a.lv[a.lc].ny * a.lv[a.lc].nx;
  const bool nf = a.lv[a.lc].cx != nullptr;
  size_t low = 0, all = 0;
  for (int l = a.lc; l < a.nl; ++l) {
    const size_t c = (size_t)a.lv[l].ny * a.lv[l].nx;
    all += c;
    if (l > a.lc) low += c;
  }
  if (large) return 3 * all * sizeof(T);
  const size_t nd = a.nl - a.lc;
  return (2 * (top + 1) + low + nd + (nf ? 4 * low : low + nd)) * sizeof(T) + all;
}
template size_t coarse_lds_bytes<float>(const CoarseArgs<float>&, bool);
template size_t coarse_lds_bytes<double>(const CoarseArgs<double>&, bool);

template <typename T, int KIND>
void launch_coarse(const CoarseArgs<T>& ca, hipStream_t s) {
  const int n = ca.lv[ca.lc].ny * ca.lv[ca.lc].nx;
  const size_t lds = coarse_lds_bytes(ca, false);
  const dim3 one(1), block(kCoarseThreads);
  if (n <= kCoarseThreads)
    hipLaunchKernelGGL((mg_coarse_lds_kernel<T, KIND, 1>), one, block, lds, s, ca);
  else if (n <= 2 * kCoarseThreads)
    hipLaunchKernelGGL((mg_coarse_lds_kernel<T, KIND, 2>), one, block, lds, s, ca);
  else
    hipLaunchKernelGGL((mg_coarse_lds_kernel<T, KIND, 4>), one, block, lds, s, ca);
}
template void launch_coarse<float, kNoflux>(const CoarseArgs<float>&, hipStream_t);
template void launch_coarse<float, kDirichlet>(const CoarseArgs<float>&, hipStream_t);
template void launch_coarse<double, kNoflux>(const CoarseArgs<double>&, hipStream_t);
template void launch_coarse<double, kDirichlet>(const CoarseArgs<double>&, hipStream_t);

template <int KIND>
void launch_coarse_batch(const CoarseArgs<float>* args, int n, int64_t cells, size_t lds,
                         hipStream_t s) {
  const dim3 grid(n), block(kCoarseThreads);
  if (cells <= kCoarseThreads)
    hipLaunchKernelGGL((mg_coarse_batch_kernel<float, KIND, 1>), grid, block, lds, s, args);
  else if (cells <= kCoarseCells)
    hipLaunchKernelGGL((mg_coarse_batch_kernel<float, KIND, 4>), grid, block, lds, s, args);
  else
    hipLaunchKernelGGL((mg_coarse_large_batch_kernel<float, KIND>), grid, block, lds, s, args);
}
template void launch_coarse_batch<kNoflux>(const CoarseArgs<float>*, int, int64_t, size_t,
                                           hipStream_t);
template void launch_coarse_batch<kDirichlet>(const CoarseArgs<float>*, int, int64_t, size_t,
                                              hipStream_t);

template <typename T, int KIND>
static void coarse_attributes() {
  const int big = (int)kCoarseLdsMax;
  for (const void* f : {(const void*)mg_coarse_lds_kernel<T, KIND, 1>,
                        (const void*)mg_coarse_lds_kernel<T, KIND, 2>,
                        (const void*)mg_coarse_lds_kernel<T, KIND, 4>})
    (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, big);
  if constexpr (sizeof(T) == 4) {
    for (const void* f : {(const void*)mg_coarse_batch_kernel<T, KIND, 1>,
                          (const void*)mg_coarse_batch_kernel<T, KIND, 4>,
                          (const void*)mg_coarse_large_batch_kernel<T, KIND>})
      (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, big);
  }
}
void coarse_lds_attributes() {
  static bool done = false;
  if (done) return;
  done = true;
  coarse_attributes<float, kNoflux>();
  coarse_attributes<float, kDirichlet>();
  coarse_attributes<double, kNoflux>();
  coarse_attributes<double, kDirichlet>();
}

}  // namespace fvx
