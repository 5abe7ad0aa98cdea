// Single-workgroup coarse V-cycle (levels lc .. nl-1 of a hierarchy): from a
// zero guess at level lc (preconditioner use) or the guess in levels[lc].u;
// the result goes to levels[lc].u.
#pragma once

#include "mg_level.hpp"

namespace fvx {

// Per-sweep weights the coarse kernel carries for each leg (sweeps past the
// last take the last weight).
constexpr int kMaxW = 8;
// Cells at or below which a level is handled by the coarse single-workgroup kernel.
constexpr int kCoarseCells = 64 * 64;
// Dynamic LDS available to the coarse kernels: 160 KB less their static
// offset table (3 x 16 ints).
constexpr size_t kCoarseLdsMax = 160 * 1024 - 3 * 16 * sizeof(int);

template <typename T>
struct CoarseArgs {
  LevelDev<T> lv[16];
  int lc, nl, n_pre, n_post, n_coarse;
  int nonzero_init;  // level lc starts from lv[lc].u instead of zero
  T w[3][kMaxW];  // sweep weights: pre-smoothing, post-smoothing, bottom
  const int* done;
};

// Dynamic LDS of one hierarchy's coarse levels (``large``: in a batch with a
// level lc over kCoarseCells, whose kernel keeps u, t and b of every level).
template <typename T>
size_t coarse_lds_bytes(const CoarseArgs<T>& a, bool large);
// One hierarchy whose level lc has at most kCoarseCells cells.
template <typename T, int KIND>
void launch_coarse(const CoarseArgs<T>& ca, hipStream_t s);
// n hierarchies (device array ``args``), one workgroup each; ``cells``: the
// largest level lc among them, lds: the largest coarse_lds_bytes.
template <int KIND>
void launch_coarse_batch(const CoarseArgs<float>* args, int n, int64_t cells, size_t lds,
                         hipStream_t s);
// Allow the coarse kernels the full 160 KB of LDS (once per process).
void coarse_lds_attributes();

}  // namespace fvx
