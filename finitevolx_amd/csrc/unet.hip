// Learned preconditioner: a bias-free convolutional U-Net (3x3 convs, 2x2
// average pooling, nearest upsampling, additive skips) with BF16 weights and
// activations and FP32 accumulation on CDNA4 matrix cores.  No reference
// counterpart; the CPU oracle is oracle/unet.py.
//
// Layout: activations channels-last (H, W, C) bf16, C a multiple of 16 except
// the 1-channel input / output handled by dedicated FP32 kernels.  Convs with
// Cin, Cout multiples of 16 are implicit GEMMs on
// v_mfma_f32_16x16x16_bf16: M = Cout, N = 16 pixels of a row, K = 16
// input channels of one tap; a workgroup owns a tile of 4 rows whose input
// (+1 halo, optionally read through nearest upsampling) is staged in LDS;
// weights are pre-packed into per-lane MFMA fragments.

#include <cmath>
#include <cstring>
#include <vector>

#include "fvx_common.hpp"

namespace fvx {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

constexpr int kUTw = 64, kUTh = 4, kUThreads = 256;

// ---------------------------------------------------------------------------
// Weight packing: fp32 w[9][Co][Ci] -> bf16 fragments
//   wp[((tap * COB + cob) * CIB + cib) * 64 + lane][i] =
//     W(tap, o = cob*16 + lane%16, c = cib*16 + 4*(lane/16) + i)
// with W(tap, o, c) = w[tap][o][c], or for the data gradient
// W(tap, o, c) = w[8 - tap][c][o] (flipped taps, swapped channels).
// ---------------------------------------------------------------------------
__global__ void pack_weights_kernel(const float* __restrict__ w, uint16_t* __restrict__ wp,
                                    int Co, int Ci, int flip) {
  // Co, Ci are the packed (output, input) channel counts.
  const int COB = Co / 16, CIB = Ci / 16;
  const int total = 9 * COB * CIB * 64 * 4;
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < total; e += gridDim.x * blockDim.x) {
    const int i = e & 3, lane = (e >> 2) & 63;
    int r = e >> 8;
    const int cib = r % CIB;
    r /= CIB;
    const int cob = r % COB;
    const int tap = r / COB;
    const int o = cob * 16 + (lane & 15), c = cib * 16 + 4 * (lane >> 4) + i;
    float v;
    if (!flip) v = w[((int64_t)tap * Co + o) * Ci + c];
    else v = w[((int64_t)(8 - tap) * Ci + c) * Co + o];  // source is w[9][Ci_src=Co][Co_src=Ci]
    wp[e] = f2bf(v);
  }
}

// ---------------------------------------------------------------------------
// 3x3 conv on matrix cores.  out = epi(sum_tap W x), epi: + skip, relu,
// * (maskt > 0).  ups: x is (H/2, W/2) and read through nearest upsampling.
//
// A workgroup owns a tile of 16 NB x 4 pixels; its COB * RG waves take one
// block of 16 output channels and 4 / RG rows each.  Most layers hold too little
// work to be bound by anything but latency (64 -> 64 channels at 64^2: 36
// matrix instructions per SIMD; large fields come to the VALU, 16 -> 16 at 1024^2
// 0.68 of its issue peak, matrix cores 0.18), so a launch is arranged as one round
// of loads: every wave requests its 9 CIB weight fragments (each reused on its
// rows x NB pixel blocks) and its share of the input tile together, then the
// tile goes to LDS (pixel pitch Cin + 8: the 16 pixels of a fragment read lie
// on different banks; the four channel groups still meet, conflicts take 0.1 to
// 0.2 of the cycles below 64 channels) and the matrix instructions run from
// registers and LDS.  NB = 1 or 2 (conv_launch).  Measured: 64 -> 64 channels at
// 64^2 7.5 us, 48 -> 48 at 128^2 6.5 us, 16 -> 16 at 512^2 9.0 us (one wave per row with the weights fetched between the matrix instructions:
// 31.5, 23.8 and 14.5 us).
// ---------------------------------------------------------------------------
constexpr int conv_row_groups(int cob) { return cob == 1 ? 4 : cob == 2 ? 2 : 1; }
constexpr int conv_threads(int cob) { return 64 * cob * conv_row_groups(cob); }

template <int COB, int CIB, int NB>
__global__ __launch_bounds__(conv_threads(COB)) void conv_mfma_kernel(
    const uint16_t* __restrict__ x, const bf16x4* __restrict__ wp, uint16_t* __restrict__ out,
    const uint16_t* __restrict__ skip, const uint16_t* __restrict__ maskt, int relu, int ups, int H,
    int W, int tiles_x, int ntiles, const int* __restrict__ guard) {
  if (guard && *guard) return;
  constexpr int RG = conv_row_groups(COB), RPW = kUTh / RG, NT = conv_threads(COB);
  constexpr int Cin = CIB * 16, Cout = COB * 16, SW = 16 * NB + 2, PITCH = Cin + 8;
  constexpr int CPP = Cin / 8;  // 16-byte chunks per pixel
  constexpr int NCH = (kUTh + 2) * SW * CPP, PER = (NCH + NT - 1) / NT;
  __shared__ __align__(16) uint16_t sx[(kUTh + 2) * SW * PITCH];
  const int t = xcd_swizzle(blockIdx.x, ntiles);
  const int i0 = (t % tiles_x) * (16 * NB), j0 = (t / tiles_x) * kUTh;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cob = wave % COB, r0 = (wave / COB) * RPW;
  const int lrow = lane & 15, lgrp = lane >> 4;
  const int Wx = W >> ups;

  bf16x4 afrag[9][CIB];
#pragma unroll
  for (int tap = 0; tap < 9; ++tap)
#pragma unroll
    for (int cib = 0; cib < CIB; ++cib)
      afrag[tap][cib] = wp[((tap * COB + cob) * CIB + cib) * 64 + lane];
  uint4 st[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = tid + k * NT, pix = c / CPP, c8 = c % CPP;
    const int gy = j0 - 1 + pix / SW, gx = i0 - 1 + pix % SW;
    st[k] = make_uint4(0u, 0u, 0u, 0u);
    if (c < NCH && gy >= 0 && gy < H && gx >= 0 && gx < W)
      st[k] = *reinterpret_cast<const uint4*>(
          x + ((int64_t)(gy >> ups) * Wx + (gx >> ups)) * Cin + 8 * c8);
  }
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int c = tid + k * NT;
    if (c < NCH) *reinterpret_cast<uint4*>(sx + (c / CPP) * PITCH + 8 * (c % CPP)) = st[k];
  }
  __syncthreads();

  f32x4 acc[RPW][NB];
#pragma unroll
  for (int r = 0; r < RPW; ++r)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[r][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int tap = 0; tap < 9; ++tap)
#pragma unroll
    for (int cib = 0; cib < CIB; ++cib)
#pragma unroll
      for (int r = 0; r < RPW; ++r)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const int pix = (r0 + r + tap / 3) * SW + nb * 16 + lrow + tap % 3;
          const bf16x4 b =
              *reinterpret_cast<const bf16x4*>(sx + pix * PITCH + cib * 16 + 4 * lgrp);
          acc[r][nb] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(afrag[tap][cib], b, acc[r][nb], 0,
                                                                 0, 0);
        }

#pragma unroll
  for (int r = 0; r < RPW; ++r) {
    const int gy = j0 + r0 + r;
    if (gy >= H) continue;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int gx = i0 + nb * 16 + lrow;
      if (gx >= W) continue;
      const int64_t o = ((int64_t)gy * W + gx) * Cout + cob * 16 + 4 * lgrp;
      float v[4] = {acc[r][nb][0], acc[r][nb][1], acc[r][nb][2], acc[r][nb][3]};
      if (skip) {
        const uint2 k = *reinterpret_cast<const uint2*>(skip + o);
        v[0] += bf2f((uint16_t)(k.x & 0xffffu));
        v[1] += bf2f((uint16_t)(k.x >> 16));
        v[2] += bf2f((uint16_t)(k.y & 0xffffu));
        v[3] += bf2f((uint16_t)(k.y >> 16));
      }
      if (relu) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = fmaxf(v[i], 0.f);
      }
      if (maskt) {
        const uint2 k = *reinterpret_cast<const uint2*>(maskt + o);
        v[0] = bf2f((uint16_t)(k.x & 0xffffu)) > 0.f ? v[0] : 0.f;
        v[1] = bf2f((uint16_t)(k.x >> 16)) > 0.f ? v[1] : 0.f;
        v[2] = bf2f((uint16_t)(k.y & 0xffffu)) > 0.f ? v[2] : 0.f;
        v[3] = bf2f((uint16_t)(k.y >> 16)) > 0.f ? v[3] : 0.f;
      }
      *reinterpret_cast<uint2*>(out + o) =
          make_uint2((uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16),
                     (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16));
    }
  }
}

// ---------------------------------------------------------------------------
// Weight gradient on matrix cores: dW[tap][co][ci] += sum_p gy[p][co] x[p+tap][ci]
// (x read through upsampling when UPS): M = 16 output channels, N = 16 input
// channels, K = 32 pixels of a row.
//
// The pixels are the contraction, so each tile (64 x 4 pixels, x with a one
// pixel halo) is transposed into LDS as [channel][row][column]: an A fragment
// is one 16-byte read, and one 16-byte and one 4-byte read give the B
// fragments of all three taps of a row (the window shifted by 0, 1, 2
// pixels with v_alignbit).  The channel pitches put the 16 channels of a
// fragment read on different banks.  The 4 / RS waves of a row group share
// out the (co, ci) block pairs, PW each, with the nine tap accumulators in
// registers over all tiles of the block; with one or two pairs the rows are
// split over RS groups instead and summed in LDS at the end.  Every block
// writes its own fp32 slot of ``part`` once; reduce_slots_kernel sums them.
// Bound: reading x and gy (16 channels: 16.8 MB at 512^2, ~3 us) and the
// transposing LDS writes.  Measured: 16 -> 16 channels at 512^2 11 us, 48 -> 48
// at 128^2 9.5 us (112 us each with 64 blocks gathering the fragments two bytes
// at a time and adding every tile to the slot in memory; 17 with one item of a
// tile at a time and a block per tile), 64 -> 64 at 64^2 9.5 us (21).
// ---------------------------------------------------------------------------
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kWXRow = 72, kWXPitch = (kUTh + 2) * kWXRow + 8;  // x: elements per row / channel
constexpr int kWGPitch = kUTh * kUTw + 24;                      // gy: elements per channel

// 4 pixels x 4 channels (one uint2 of channels per pixel) -> 4 uint2 of pixels.
__device__ __forceinline__ void transpose4(const uint2 (&p)[4], uint2 (&c)[4]) {
  c[0] = make_uint2((p[0].x & 0xffffu) | (p[1].x << 16), (p[2].x & 0xffffu) | (p[3].x << 16));
  c[1] = make_uint2((p[0].x >> 16) | (p[1].x & 0xffff0000u),
                    (p[2].x >> 16) | (p[3].x & 0xffff0000u));
  c[2] = make_uint2((p[0].y & 0xffffu) | (p[1].y << 16), (p[2].y & 0xffffu) | (p[3].y << 16));
  c[3] = make_uint2((p[0].y >> 16) | (p[1].y & 0xffff0000u),
                    (p[2].y >> 16) | (p[3].y & 0xffff0000u));
}

// items items of 4 pixels x 4 channels: load(item, pixels), transposed,
// store(item, channels), the loads of two items a thread in flight together
// (one after the other, each item was a memory latency).
template <typename Load, typename Store>
__device__ __forceinline__ void stage_items(int items, Load load, Store store) {
  for (int k = threadIdx.x; k < items; k += 2 * kUThreads) {
    uint2 p[2][4], c[4];
    const int k1 = k + kUThreads;
    load(k, p[0]);
    load(min(k1, items - 1), p[1]);
    transpose4(p[0], c);
    store(k, c);
    if (k1 < items) {
      transpose4(p[1], c);
      store(k1, c);
    }
  }
}

template <int PW, int RS, bool UPS>
__global__ __launch_bounds__(kUThreads) void conv_bwdw_mfma_kernel(
    const uint16_t* __restrict__ x, int Cin, const uint16_t* __restrict__ gy, int Cout, int cobn,
    float* __restrict__ part, int H, int W, int tiles_x, int ntiles) {
  extern __shared__ __align__(16) uint16_t smem[];
  uint16_t* sx = smem;                           // [Cin][TH + 2][kWXRow]
  uint16_t* sg = smem + (int64_t)Cin * kWXPitch;  // [16 cobn][TH][TW]
  constexpr int NWP = 4 / RS, ROWS = kUTh / RS;
  const int CIB = Cin / 16, NP = cobn * CIB, cob0 = blockIdx.y * cobn;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wp = wave % NWP, rs = wave / NWP;
  const int lrow = lane & 15, lgrp = lane >> 4;
  const int Wx = UPS ? W / 2 : W;
  f32x4 acc[PW][9];
#pragma unroll
  for (int k = 0; k < PW; ++k)
#pragma unroll
    for (int q = 0; q < 9; ++q) acc[k][q] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
    const int i0 = (t % tiles_x) * kUTw, j0 = (t / tiles_x) * kUTh;
    __syncthreads();
    const int c4x = Cin / 4, c4g = 4 * cobn;
    stage_items(
        (kUTh + 2) * 17 * c4x,
        [&](int k, uint2(&px)[4]) {
          const int c4 = k % c4x, u = k / c4x, g = u % 17, gyy = j0 - 1 + u / 17;
          const int cy = min(max(gyy, 0), H - 1);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int gxx = i0 - 1 + 4 * g + e, cx = min(max(gxx, 0), W - 1);
            const int sy = UPS ? (cy >> 1) : cy, sxx = UPS ? (cx >> 1) : cx;
            px[e] = *reinterpret_cast<const uint2*>(x + ((int64_t)sy * Wx + sxx) * Cin + 4 * c4);
            if (cy != gyy || cx != gxx) px[e] = make_uint2(0u, 0u);
          }
        },
        [&](int k, const uint2(&ch)[4]) {
          const int c4 = k % c4x, u = k / c4x, g = u % 17, ry = u / 17;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            *reinterpret_cast<uint2*>(sx + (4 * c4 + e) * kWXPitch + ry * kWXRow + 4 * g) = ch[e];
        });
    stage_items(
        kUTh * (kUTw / 4) * c4g,
        [&](int k, uint2(&px)[4]) {
          const int c4 = k % c4g, u = k / c4g, g = u % (kUTw / 4), gyy = j0 + u / (kUTw / 4);
          const int cy = min(gyy, H - 1);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int gxx = i0 + 4 * g + e, cx = min(gxx, W - 1);
            px[e] = *reinterpret_cast<const uint2*>(gy + ((int64_t)cy * W + cx) * Cout +
                                                    16 * cob0 + 4 * c4);
            if (cy != gyy || cx != gxx) px[e] = make_uint2(0u, 0u);
          }
        },
        [&](int k, const uint2(&ch)[4]) {
          const int c4 = k % c4g, u = k / c4g, g = u % (kUTw / 4), ry = u / (kUTw / 4);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            *reinterpret_cast<uint2*>(sg + (4 * c4 + e) * kWGPitch + ry * kUTw + 4 * g) = ch[e];
        });
    __syncthreads();
    for (int rk = 0; rk < 2 * ROWS; ++rk) {
      const int r = rs * ROWS + (rk >> 1), col = 32 * (rk & 1) + 8 * lgrp;
#pragma unroll
      for (int k = 0; k < PW; ++k) {
        const int p = wp + NWP * k;
        if (p < NP) {
          const int cob = p / CIB, cib = p - cob * CIB;
          const bf16x8 a =
              *reinterpret_cast<const bf16x8*>(sg + (cob * 16 + lrow) * kWGPitch + r * kUTw + col);
#pragma unroll
          for (int ky = 0; ky < 3; ++ky) {
            const uint16_t* b =
                sx + (cib * 16 + lrow) * kWXPitch + (r + ky) * kWXRow + col;
            const uint4 lo = *reinterpret_cast<const uint4*>(b);
            const uint32_t hi = *reinterpret_cast<const uint32_t*>(b + 8);
            const uint4 b1 = make_uint4(__builtin_amdgcn_alignbit(lo.y, lo.x, 16),
                                        __builtin_amdgcn_alignbit(lo.z, lo.y, 16),
                                        __builtin_amdgcn_alignbit(lo.w, lo.z, 16),
                                        __builtin_amdgcn_alignbit(hi, lo.w, 16));
            const uint4 b2 = make_uint4(lo.y, lo.z, lo.w, hi);
            acc[k][3 * ky] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                a, __builtin_bit_cast(bf16x8, lo), acc[k][3 * ky], 0, 0, 0);
            acc[k][3 * ky + 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                a, __builtin_bit_cast(bf16x8, b1), acc[k][3 * ky + 1], 0, 0, 0);
            acc[k][3 * ky + 2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                a, __builtin_bit_cast(bf16x8, b2), acc[k][3 * ky + 2], 0, 0, 0);
          }
        }
      }
    }
  }
  if constexpr (RS > 1) {
    f32x4* sr = reinterpret_cast<f32x4*>(smem);  // [(RS - 1) * NWP][PW * 9][64]
    __syncthreads();
    if (rs > 0) {
#pragma unroll
      for (int k = 0; k < PW; ++k)
#pragma unroll
        for (int q = 0; q < 9; ++q)
          sr[(((rs - 1) * NWP + wp) * PW * 9 + k * 9 + q) * 64 + lane] = acc[k][q];
    }
    __syncthreads();
    if (rs > 0) return;
    for (int o = 0; o < RS - 1; ++o)
#pragma unroll
      for (int k = 0; k < PW; ++k)
#pragma unroll
        for (int q = 0; q < 9; ++q)
          acc[k][q] += sr[((o * NWP + wp) * PW * 9 + k * 9 + q) * 64 + lane];
  }
  float* mine = part + (int64_t)blockIdx.x * 9 * Cout * Cin;
#pragma unroll
  for (int k = 0; k < PW; ++k) {
    const int p = wp + NWP * k;
    if (p >= NP) continue;
    const int cob = p / CIB, cib = p - cob * CIB;
#pragma unroll
    for (int q = 0; q < 9; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        mine[((int64_t)q * Cout + (cob0 + cob) * 16 + 4 * lgrp + i) * Cin + cib * 16 + lrow] = acc[k][q][i];
  }
}

// out[e] += sum over slots of part[g][e] for every layer of a backward pass in
// one launch (14 of them took 5 us each at the default network), 64 elements a
// block: 16 wavefronts take every 16th slot (independent loads in flight; with
// one thread per element the 64 slots were a 15 us chain), then sum in LDS in
// wave order.
constexpr int kRedWaves = 16, kMaxLayers = 31;  // 8 levels: 16 + 14 + 1
struct RedTable {
  int layers = 0, blocks = 0;
  struct {
    const float* part;
    float* out;
    int nslot, n, block0;
  } l[kMaxLayers];
};
__global__ __launch_bounds__(64 * kRedWaves) void reduce_slots_kernel(RedTable t) {
  __shared__ float red[kRedWaves][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int k = 0;
  while (k + 1 < t.layers && (int)blockIdx.x >= t.l[k + 1].block0) ++k;
  const float* part = t.l[k].part;
  float* out = t.l[k].out;
  const int nslot = t.l[k].nslot, n = t.l[k].n;
  const int e = ((int)blockIdx.x - t.l[k].block0) * 64 + lane;
  float s = 0.f;
  if (e < n) {
#pragma unroll 8
    for (int g = wave; g < nslot; g += kRedWaves) s += part[(int64_t)g * n + e];
  }
  red[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && e < n) {
    float v = 0.f;
#pragma unroll
    for (int q = 0; q < kRedWaves; ++q) v += red[q][lane];
    out[e] += v;
  }
}

// ---------------------------------------------------------------------------
// 1-channel input / output layers (FP32 arithmetic).
// ---------------------------------------------------------------------------
// out[p][c] = relu(sum_tap w[tap][c] r[p+tap]),  r fp32 (H, W), w fp32 [9][C]
__global__ void conv_first_kernel(const float* __restrict__ r, const float* __restrict__ w, int C,
                                  uint16_t* __restrict__ out, int H, int W,
                                  const int* __restrict__ guard) {
  if (guard && *guard) return;
  const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
  if (i >= W || j >= H) return;
  float nb[9];
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    const int y = j + t / 3 - 1, x = i + t % 3 - 1;
    nb[t] = (y >= 0 && y < H && x >= 0 && x < W) ? r[(int64_t)y * W + x] : 0.f;
  }
  const int64_t p = (int64_t)j * W + i;
  // 8 channels per 16-byte store (C is a multiple of 16).
  for (int c8 = 0; c8 < C; c8 += 8) {
    uint32_t pk[4];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      float s0 = 0.f, s1 = 0.f;
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        s0 += w[t * C + c8 + 2 * h] * nb[t];
        s1 += w[t * C + c8 + 2 * h + 1] * nb[t];
      }
      pk[h] = (uint32_t)f2bf(fmaxf(s0, 0.f)) | ((uint32_t)f2bf(fmaxf(s1, 0.f)) << 16);
    }
    *reinterpret_cast<uint4*>(out + p * C + c8) = make_uint4(pk[0], pk[1], pk[2], pk[3]);
  }
}

// y[p] = scale * sum_tap sum_c w[tap][c] d[p+tap][c]; optional mask multiply.
// Each pixel's channels are read 8 at a time (16-byte loads).
template <typename TO>
__global__ void conv_last_kernel(const uint16_t* __restrict__ d, const float* __restrict__ w,
                                 int C, TO* __restrict__ y, int64_t ld_y, int H, int W,
                                 const float* __restrict__ scale, const uint8_t* __restrict__ mask,
                                 const int* __restrict__ guard) {
  if (guard && *guard) return;
  const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
  if (i >= W || j >= H) return;
  float s = 0.f;
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    const int yy = j + t / 3 - 1, xx = i + t % 3 - 1;
    if (yy < 0 || yy >= H || xx < 0 || xx >= W) continue;
    const uint16_t* dp = d + ((int64_t)yy * W + xx) * C;
    for (int c8 = 0; c8 < C; c8 += 8) {
      const uint4 v = *reinterpret_cast<const uint4*>(dp + c8);
      const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        s += w[t * C + c8 + 2 * h] * bf2f((uint16_t)(u[h] & 0xffffu));
        s += w[t * C + c8 + 2 * h + 1] * bf2f((uint16_t)(u[h] >> 16));
      }
    }
  }
  if (scale) s *= *scale;
  if (mask && !mask[(int64_t)j * W + i]) s = 0.f;
  y[(int64_t)j * ld_y + i] = (TO)s;
}

// g_d[q][c] = (d[q][c] > 0) * sum_tap w[tap][c] gy[q - tap]; 8 channels per
// 16-byte load and store (one channel at a time: 24 us at 512^2, 16 channels).
__global__ void conv_last_bwd_data_kernel(const float* __restrict__ gy, const float* __restrict__ w,
                                          int C, const uint16_t* __restrict__ d,
                                          uint16_t* __restrict__ gd, int H, int W) {
  const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
  if (i >= W || j >= H) return;
  float g[9];
#pragma unroll
  for (int t = 0; t < 9; ++t) {
    const int y = j - (t / 3 - 1), x = i - (t % 3 - 1);
    g[t] = (y >= 0 && y < H && x >= 0 && x < W) ? gy[(int64_t)y * W + x] : 0.f;
  }
  const int64_t q = (int64_t)j * W + i;
  for (int c8 = 0; c8 < C; c8 += 8) {
    const uint4 dv = *reinterpret_cast<const uint4*>(d + q * C + c8);
    const uint32_t du[4] = {dv.x, dv.y, dv.z, dv.w};
    uint32_t pk[4];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      float s0 = 0.f, s1 = 0.f;
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        s0 += w[t * C + c8 + 2 * h] * g[t];
        s1 += w[t * C + c8 + 2 * h + 1] * g[t];
      }
      s0 = bf2f((uint16_t)(du[h] & 0xffffu)) > 0.f ? s0 : 0.f;
      s1 = bf2f((uint16_t)(du[h] >> 16)) > 0.f ? s1 : 0.f;
      pk[h] = (uint32_t)f2bf(s0) | ((uint32_t)f2bf(s1) << 16);
    }
    *reinterpret_cast<uint4*>(gd + q * C + c8) = make_uint4(pk[0], pk[1], pk[2], pk[3]);
  }
}

// Per-block partial sums of the one-channel layers' weight gradients, FP32:
// dW[tap][c] = sum_q sc[q][c] s1[q - sgn tap] (sgn = +1: s1 is the gradient of
// the output layer and sc its input; sgn = -1: s1 is the input field and sc
// the gradient of the first layer).  A thread owns 8 channels of every
// (256 * 8 / C)-th pixel of its block: one 16-byte load of sc and nine of s1
// feed its 72 register sums, where one pass over both fields per (tap, c)
// took 846 us at 512^2 with 16 channels (now 10 us; 15 with a select on every
// tap of every pixel, 34 with 216 lane moves in the sums over lanes).  part: [nblk][9 * C].
__global__ __launch_bounds__(256) void edge_bwdw_kernel(const float* __restrict__ s1,
                                                        const uint16_t* __restrict__ sc, int C,
                                                        int sgn, float* __restrict__ part, int H,
                                                        int W) {
  __shared__ float red[4][9 * 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int cg = C / 8;  // threads per pixel: 2, 4, 6 or 8
  const int ppw = 64 / cg;  // pixels per wavefront pass (6 groups: 10, four lanes idle)
  const int c8 = lane % cg, pl = lane / cg;
  const int64_t N = (int64_t)H * W;
  const int64_t per = (N + gridDim.x - 1) / gridDim.x;
  const int64_t p0 = (int64_t)blockIdx.x * per, p1 = min(N, p0 + per);
  float acc[9][8];
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int h = 0; h < 8; ++h) acc[t][h] = 0.f;
  if (pl < ppw) {
    for (int64_t p = p0 + wave * ppw + pl; p < p1; p += 4 * ppw) {
      const int j = (int)((uint32_t)p / (uint32_t)W), i = (int)((uint32_t)p % (uint32_t)W);
      const uint4 v = *reinterpret_cast<const uint4*>(sc + p * C + 8 * c8);
      const uint32_t u[4] = {v.x, v.y, v.z, v.w};
      float f[8];
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        f[2 * h] = bf2f((uint16_t)(u[h] & 0xffffu));
        f[2 * h + 1] = bf2f((uint16_t)(u[h] >> 16));
      }
      float g[9];
      uint32_t in = 0;
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        const int y = j - sgn * (t / 3 - 1), x = i - sgn * (t % 3 - 1);
        const int cy = min(max(y, 0), H - 1), cx = min(max(x, 0), W - 1);
        g[t] = s1[(int64_t)cy * W + cx];
        in |= cy == y && cx == x ? 1u << t : 0u;
      }
      // (outside, no product: 0 times an overflowed value would be NaN)
      if (__ballot(in != 0x1ff) == 0) {
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
          for (int h = 0; h < 8; ++h) acc[t][h] += g[t] * f[h];
      } else {
#pragma unroll
        for (int t = 0; t < 9; ++t)
#pragma unroll
          for (int h = 0; h < 8; ++h) acc[t][h] += (in >> t) & 1 ? g[t] * f[h] : 0.f;
      }
    }
  }
  // Sum over the lanes of one channel group (stride cg).  Power-of-two groups:
  // three butterfly steps that hand half of the sums to the other lane each
  // (channels 4, 2, 1: 63 lane moves instead of 216), then plain ones; lane l
  // ends with the nine taps of channel 4 l5 + 2 l4 + l3 of its group.  Six
  // groups through their first lanes.
  if (cg != 6) {
    float r4[9][4], r2[9][2], r1[9];
    const bool h5 = lane & 32, h4 = lane & 16, h3 = lane & 8;
#pragma unroll
    for (int t = 0; t < 9; ++t) {
#pragma unroll
      for (int h = 0; h < 4; ++h)
        r4[t][h] = (h5 ? acc[t][h + 4] : acc[t][h]) +
                   __shfl_xor(h5 ? acc[t][h] : acc[t][h + 4], 32);
#pragma unroll
      for (int h = 0; h < 2; ++h)
        r2[t][h] = (h4 ? r4[t][h + 2] : r4[t][h]) + __shfl_xor(h4 ? r4[t][h] : r4[t][h + 2], 16);
      r1[t] = (h3 ? r2[t][1] : r2[t][0]) + __shfl_xor(h3 ? r2[t][0] : r2[t][1], 8);
      for (int o = 4; o >= cg; o >>= 1) r1[t] += __shfl_xor(r1[t], o);
    }
    const int h = (h5 ? 4 : 0) + (h4 ? 2 : 0) + (h3 ? 1 : 0);
    if ((lane & 7) < cg) {
#pragma unroll
      for (int t = 0; t < 9; ++t) red[wave][t * C + 8 * c8 + h] = r1[t];
    }
  } else {
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int h = 0; h < 8; ++h) {
        float r = acc[t][h];
        for (int k = 1; k < 10; ++k) r += __shfl(acc[t][h], min(lane + 6 * k, 63));
        if (lane < cg) red[wave][t * C + 8 * c8 + h] = r;
      }
  }
  __syncthreads();
  for (int e = tid; e < 9 * C; e += 256)
    part[(int64_t)blockIdx.x * 9 * C + e] = ((red[0][e] + red[1][e]) + red[2][e]) + red[3][e];
}

// ---------------------------------------------------------------------------
// Pooling and gradient combination (bf16 HWC).
// ---------------------------------------------------------------------------
__global__ void pool2_kernel(const uint16_t* __restrict__ in, uint16_t* __restrict__ out, int H,
                             int W, int C, const int* __restrict__ guard) {  // H, W: output dims
  if (guard && *guard) return;
  const int64_t n = (int64_t)H * W * C;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int c = (int)(e % C);
    const int64_t p = e / C;
    const int I = (int)(p % W), J = (int)(p / W);
    const int64_t W2 = 2 * W;
    const float s = bf2f(in[((2 * J) * W2 + 2 * I) * C + c]) + bf2f(in[((2 * J) * W2 + 2 * I + 1) * C + c]) +
                    bf2f(in[((2 * J + 1) * W2 + 2 * I) * C + c]) +
                    bf2f(in[((2 * J + 1) * W2 + 2 * I + 1) * C + c]);
    out[e] = f2bf(0.25f * s);
  }
}

// out[J][I][c] = (h[J][I][c] > 0) * sum_{a,b} g[2J+a][2I+b][c]   (up2 backward + relu mask)
__global__ void upbwd_mask_kernel(const uint16_t* __restrict__ g, const uint16_t* __restrict__ h,
                                  uint16_t* __restrict__ out, int H, int W, int C) {
  const int64_t n = (int64_t)H * W * C;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int c = (int)(e % C);
    const int64_t p = e / C;
    const int I = (int)(p % W), J = (int)(p / W);
    const int64_t W2 = 2 * W;
    const float s = bf2f(g[((2 * J) * W2 + 2 * I) * C + c]) + bf2f(g[((2 * J) * W2 + 2 * I + 1) * C + c]) +
                    bf2f(g[((2 * J + 1) * W2 + 2 * I) * C + c]) +
                    bf2f(g[((2 * J + 1) * W2 + 2 * I + 1) * C + c]);
    out[e] = f2bf(bf2f(h[e]) > 0.f ? s : 0.f);
  }
}

// out[j][i][c] = (h[j][i][c] > 0) * (skip[j][i][c] + 0.25 gc[j/2][i/2][c])  (pool backward)
__global__ void poolbwd_add_mask_kernel(const uint16_t* __restrict__ skip,
                                        const uint16_t* __restrict__ gc,
                                        const uint16_t* __restrict__ h, uint16_t* __restrict__ out,
                                        int H, int W, int C) {
  const int64_t n = (int64_t)H * W * C;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int c = (int)(e % C);
    const int64_t p = e / C;
    const int i = (int)(p % W), j = (int)(p / W);
    const float v = (skip ? bf2f(skip[e]) : 0.f) +
                    0.25f * bf2f(gc[((int64_t)(j / 2) * (W / 2) + i / 2) * C + c]);
    out[e] = f2bf(bf2f(h[e]) > 0.f ? v : 0.f);
  }
}

// ---------------------------------------------------------------------------
// Input normalisation, loss, Adam.
// ---------------------------------------------------------------------------
// s = rms of the residual (FP64 accumulate): per-block partials, then a
// one-workgroup finish (kernel boundary in between, no device fences):
// scal[0] = 1/s (input scale), scal[1] = s * out_scale (output scale).
template <typename T>
__global__ __launch_bounds__(256) void rms_kernel(const T* __restrict__ r, int64_t ld, int H, int W,
                                                   double* __restrict__ part,
                                                   const int* __restrict__ guard) {
  if (guard && *guard) return;
  __shared__ double red[256];
  const int tid = threadIdx.x;
  double acc = 0.0;
  const int64_t N = (int64_t)H * W;
  for (int64_t p = blockIdx.x * 256 + tid; p < N; p += (int64_t)gridDim.x * 256) {
    const double v = (double)r[(p / W) * ld + p % W];
    acc += v * v;
  }
  red[tid] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (tid < s) red[tid] += red[tid + s];
    __syncthreads();
  }
  if (tid == 0) part[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void rms_finish_kernel(const double* __restrict__ part, int nb,
                                                          int64_t N, float* __restrict__ scal,
                                                          double out_scale,
                                                          const int* __restrict__ guard) {
  if (guard && *guard) return;
  __shared__ double red[256];
  const int tid = threadIdx.x;
  double acc = 0.0;
  for (int b = tid; b < nb; b += 256) acc += part[b];
  red[tid] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (tid < s) red[tid] += red[tid + s];
    __syncthreads();
  }
  if (tid == 0) {
    const double rms = sqrt(red[0] / (double)N);
    scal[0] = rms > 0.0 ? (float)(1.0 / rms) : 0.f;
    scal[1] = (float)(rms * out_scale);
  }
}

template <typename T>
__global__ void scale_in_kernel(const T* __restrict__ r, int64_t ld, int H, int W,
                                const float* __restrict__ scal, float* __restrict__ out,
                                const int* __restrict__ guard) {
  if (guard && *guard) return;
  const int i = blockIdx.x * 64 + threadIdx.x, j = blockIdx.y * 4 + threadIdx.y;
  if (i < W && j < H) out[(int64_t)j * W + i] = (float)r[(int64_t)j * ld + i] * scal[0];
}

// gy = 2 (y - e) / n  (loss = mean (y - e)^2), loss partial sums in part.
__global__ __launch_bounds__(256) void mse_grad_kernel(const float* __restrict__ y,
                                                       const float* __restrict__ e,
                                                       float* __restrict__ gy, int64_t n,
                                                       double* __restrict__ loss_acc) {
  __shared__ double red[256];
  const int tid = threadIdx.x;
  double acc = 0.0;
  for (int64_t k = blockIdx.x * 256 + tid; k < n; k += (int64_t)gridDim.x * 256) {
    const float d = y[k] - e[k];
    gy[k] = 2.f * d / (float)n;
    acc += (double)d * d;
  }
  red[tid] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (tid < s) red[tid] += red[tid + s];
    __syncthreads();
  }
  if (tid == 0) atomicAdd(loss_acc, red[0] / (double)n);
}

__global__ void adam_kernel(float* __restrict__ w, float* __restrict__ g, float* __restrict__ m,
                            float* __restrict__ v, int64_t n, float lr, float b1, float b2,
                            float eps, float bc1, float bc2, float gscale) {
  for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < n;
       k += (int64_t)gridDim.x * blockDim.x) {
    const float gk = g[k] * gscale;
    const float mk = b1 * m[k] + (1.f - b1) * gk;
    const float vk = b2 * v[k] + (1.f - b2) * gk * gk;
    m[k] = mk;
    v[k] = vk;
    w[k] -= lr * (mk / bc1) / (sqrtf(vk / bc2) + eps);
    g[k] = 0.f;
  }
}

// ---------------------------------------------------------------------------
// Network plan
// ---------------------------------------------------------------------------
struct Layer {
  int cout, cin;
  size_t off;  // offset (floats) into the master weight buffer
};

struct UNet {
  int L;                    // levels
  int ch[8];
  int H, W;                 // spatial size the buffers are sized for
  std::vector<Layer> layers;  // order: e0a e0b e1a e1b ... u_{L-2} d_{L-2} ... u0 d0 out
  size_t nweights = 0;
  float *w = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;   // fp32 master / grad / Adam
  uint16_t* wpk = nullptr;   // packed bf16 forward fragments (per layer offsets)
  uint16_t* wpkT = nullptr;  // packed flipped/transposed fragments (data gradient)
  std::vector<size_t> pk_off;
  // activations per level: x (pooled input, l > 0), h1e, e (=h2e), h1d, d
  std::vector<uint16_t*> xin, h1e, ee, h1d, dd, gA, gB, gC;
  float *rin = nullptr, *yout = nullptr, *gy = nullptr, *eref = nullptr;
  // Weight-gradient slots: of the layer with most (``widest``) in part, the
  // others' from part_off in rest, which the first backward pass allocates;
  // without rest every layer takes part and is summed before the next.
  float *part = nullptr, *rest = nullptr;
  size_t rest_elems = 0;
  int widest = 0;
  std::vector<size_t> part_off;
  double* rms_part = nullptr;
  float* scal = nullptr;
  double* loss = nullptr;
  const int* guard = nullptr;  // PCG convergence flag: kernels exit when set
  int adam_t = 0;
  std::vector<void*> allocs;
};

static int layer_index(const UNet& N, char kind, int l) {
  // e: 2l (a) / 2l+1 (b); u/d: 2L + 2*(L-2-l) (+1 for d); out: last
  if (kind == 'a') return 2 * l;
  if (kind == 'b') return 2 * l + 1;
  if (kind == 'u') return 2 * N.L + 2 * (N.L - 2 - l);
  if (kind == 'd') return 2 * N.L + 2 * (N.L - 2 - l) + 1;
  return (int)N.layers.size() - 1;
}

template <typename T>
static int dev_alloc(UNet& N, T** p, size_t n) {
  void* q = nullptr;
  FVX_HIP(hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T)));
  N.allocs.push_back(q);
  *p = (T*)q;
  return kOk;
}

static void conv_launch(const UNet& N, int li, bool transposed, const uint16_t* x, uint16_t* out,
                        const uint16_t* skip, const uint16_t* maskt, bool relu, bool ups, int H,
                        int W, hipStream_t s) {
  const Layer& Ly = N.layers[li];
  const int cout = transposed ? Ly.cin : Ly.cout, cin = transposed ? Ly.cout : Ly.cin;
  const bf16x4* wp = (const bf16x4*)((transposed ? N.wpkT : N.wpk) + N.pk_off[li]);
  // Tiles 16 pixels wide (halo 1.7x): many workgroups, which hide each other's
  // loads.  32 wide (halo 1.6x) on large fields with few output channels, which
  // are nearer the memory than the matrix cores.  us, 16 / 32 / 64 wide:
  //   16 -> 16 channels  256 x 512  7.5 /  7.5 /  7.8   512^2 10.4 /  9.0 /  9.8
  //                         1024^2 25.0 / 19.3 / 20.6  2048^2   83 /   61 /   59
  //   48 -> 32           256 x 512 13.9 / 13.3 / 14.6  1024^2 68.6 / 59.5 / 81.4
  //   32 -> 48              512^2  20.3 / 21.6 / 27.1  2048^2  286 /  241 /  318
  //   48 -> 48              512^2  24.7 / 34.7 / 50.2  2048^2  359 /  473 /  740
  //   64 -> 64              512^2  40.7 / 44.6 / 57.1  2048^2  598 /  590 /  844
  // (64 wide: one wave a SIMD with 48 and 64 channels, whose weights, accumulators
  // and staging fill its registers).
  const bool wide = cout <= 32 && cdiv(W, 64) * cdiv(H, kUTh) >= 1024;
  const int tx = cdiv(W, wide ? 32 : 16), nt = tx * cdiv(H, kUTh);
#define FVX_CONV_NB(COB, CIB, NB)                                                              \
  hipLaunchKernelGGL((conv_mfma_kernel<COB, CIB, NB>), dim3(nt), dim3(conv_threads(COB)), 0, s, x, \
                     wp, out, skip, maskt, relu ? 1 : 0, ups ? 1 : 0, H, W, tx, nt, N.guard)
#define FVX_CONV(COB, CIB)                   \
  if constexpr (COB > 2) FVX_CONV_NB(COB, CIB, 1); \
  else if (wide) FVX_CONV_NB(COB, CIB, 2);   \
  else FVX_CONV_NB(COB, CIB, 1)
#define FVX_CONV_CI(COB)                     \
  switch (cin / 16) {                        \
    case 1: FVX_CONV(COB, 1); break;         \
    case 2: FVX_CONV(COB, 2); break;         \
    case 3: FVX_CONV(COB, 3); break;         \
    default: FVX_CONV(COB, 4); break;        \
  }
  switch (cout / 16) {
    case 1: FVX_CONV_CI(1); break;
    case 2: FVX_CONV_CI(2); break;
    case 3: FVX_CONV_CI(3); break;
    default: FVX_CONV_CI(4); break;
  }
#undef FVX_CONV_CI
#undef FVX_CONV
#undef FVX_CONV_NB
}

static dim3 g2(int H, int W) { return dim3(cdiv(W, 64), cdiv(H, 4)); }
static dim3 g1(int64_t n) { return dim3((unsigned)std::min<int64_t>((n + 255) / 256, 4096)); }

// Forward pass on N.rin (already scaled); result in N.yout (fp32), unscaled.
// With last == false the output conv is left to the caller.
static int unet_forward(UNet& N, int H, int W, hipStream_t s, bool last = true) {
  const int L = N.L;
  // encoder
  for (int l = 0; l < L; ++l) {
    const int h = H >> l, w = W >> l;
    if (l == 0) {
      const Layer& a = N.layers[layer_index(N, 'a', 0)];
      hipLaunchKernelGGL(conv_first_kernel, g2(h, w), dim3(64, 4), 0, s, N.rin, N.w + a.off,
                         N.ch[0], N.h1e[0], h, w, N.guard);
    } else {
      hipLaunchKernelGGL(pool2_kernel, g1((int64_t)h * w * N.ch[l - 1]), dim3(256), 0, s,
                         N.ee[l - 1], N.xin[l], h, w, N.ch[l - 1], N.guard);
      conv_launch(N, layer_index(N, 'a', l), false, N.xin[l], N.h1e[l], nullptr, nullptr, true,
                  false, h, w, s);
    }
    conv_launch(N, layer_index(N, 'b', l), false, N.h1e[l], N.ee[l], nullptr, nullptr, true, false,
                h, w, s);
  }
  // decoder
  const uint16_t* dprev = N.ee[L - 1];
  for (int l = L - 2; l >= 0; --l) {
    const int h = H >> l, w = W >> l;
    conv_launch(N, layer_index(N, 'u', l), false, dprev, N.h1d[l], N.ee[l], nullptr, true, true, h,
                w, s);
    conv_launch(N, layer_index(N, 'd', l), false, N.h1d[l], N.dd[l], nullptr, nullptr, true, false,
                h, w, s);
    dprev = N.dd[l];
  }
  if (last) {
    const Layer& o = N.layers.back();
    hipLaunchKernelGGL((conv_last_kernel<float>), g2(H, W), dim3(64, 4), 0, s, dprev, N.w + o.off,
                       N.ch[0], N.yout, (int64_t)W, H, W, nullptr, nullptr, N.guard);
  }
  FVX_LAUNCH_CHECK();
  return kOk;
}

// Slots of layer li's weight gradient at H x W pixels: a block per tile, at most
// two per CU (each writes a slot that the reduction reads back, so more only add
// traffic) and 9.4 MB; the one-channel layers a block per 256 pixels.
constexpr int kBwdwBlocks = 512, kBwdwSplit = 256;
static int bwdw_slots(const Layer& Ly, int H, int W) {
  if (Ly.cout == 1 || Ly.cin == 1)
    return (int)std::min<int64_t>(((int64_t)H * W + 255) / 256, kBwdwBlocks);
  const size_t n = (size_t)9 * Ly.cout * Ly.cin;
  const int nt = cdiv(W, kUTw) * cdiv(H, kUTh);
  return (int)std::min<size_t>(std::min(nt, kBwdwBlocks), (size_t)64 * 9 * 64 * 64 / n);
}
static float* layer_part(const UNet& N, int li) {
  return N.rest && li != N.widest ? N.rest + N.part_off[li] : N.part;
}
static void red_flush(RedTable& t, hipStream_t s) {
  if (t.layers)
    hipLaunchKernelGGL(reduce_slots_kernel, dim3(t.blocks), dim3(64 * kRedWaves), 0, s, t);
  t = RedTable();
}
static void red_add(const UNet& N, int li, int nslot, RedTable& t, hipStream_t s) {
  const Layer& Ly = N.layers[li];
  auto& e = t.l[t.layers++];
  e.part = layer_part(N, li);
  e.out = N.g + Ly.off;
  e.nslot = nslot;
  e.n = 9 * Ly.cout * Ly.cin;
  e.block0 = t.blocks;
  t.blocks += cdiv(e.n, 64);
  if (!N.rest) red_flush(t, s);
}
// The other layers' slots, with the first backward pass (plans that only run
// forward hold none).  Under capture, where nothing can be allocated, or without
// the memory, the passes go on layer by layer.
static void take_slots(UNet& N, hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  void* p = nullptr;
  if (N.rest) return;
  if (hipStreamIsCapturing(s, &st) == hipSuccess && st == hipStreamCaptureStatusNone &&
      hipMalloc(&p, N.rest_elems * sizeof(float)) == hipSuccess) {
    N.allocs.push_back(p);
    N.rest = (float*)p;
  } else {
    (void)hipGetLastError();
  }
}

template <int PW, int RS, bool UPS>
static void launch_bwdw(float* part, const Layer& Ly, const uint16_t* x, const uint16_t* gyt, int G,
                        int cobn, int H, int W, int tx, int nt, hipStream_t s) {
  const size_t stage = ((size_t)Ly.cin * kWXPitch + (size_t)16 * cobn * kWGPitch) * sizeof(uint16_t);
  const size_t sums = (size_t)(RS - 1) * (4 / RS) * PW * 9 * 64 * sizeof(f32x4);
  hipLaunchKernelGGL((conv_bwdw_mfma_kernel<PW, RS, UPS>), dim3(G, Ly.cout / 16 / cobn),
                     dim3(kUThreads), std::max(stage, sums), s, x, Ly.cin, gyt, Ly.cout, cobn,
                     part, H, W, tx, nt);
}

static void bwdw_launch(UNet& N, int li, const uint16_t* x, const uint16_t* gyt, bool ups, int H,
                        int W, RedTable& red, hipStream_t s) {
  const Layer& Ly = N.layers[li];
  float* part = layer_part(N, li);
  const int tx = cdiv(W, kUTw), ty = cdiv(H, kUTh), nt = tx * ty;
  const int G = bwdw_slots(Ly, H, W);
  // Few tiles: a block per 16 output channels (and tile), which leaves each the
  // x tile, a share of gy and of the products.  Gradient, us, splitting never / up
  // to 64, 128, 256, 512 tiles: default network 128^2 475 / 422 426 420 430, 512^2
  // 631 / 588 588 587 583, 1024^2 1366 / 1350 1293 1266 1267; channels (32, 48)
  // 512^2 561 / 560 546 523 523, 1024^2 1786 / 1787 1733 1644 1643.
  const int cobn = G <= kBwdwSplit ? 1 : Ly.cout / 16;
  const int np = cobn * (Ly.cin / 16);  // (co, ci) block pairs of a block, 1 .. 16
#define FVX_BWDW(PW, RS)                                                          \
  (ups ? launch_bwdw<PW, RS, true>(part, Ly, x, gyt, G, cobn, H, W, tx, nt, s)       \
       : launch_bwdw<PW, RS, false>(part, Ly, x, gyt, G, cobn, H, W, tx, nt, s))
  if (np == 1) FVX_BWDW(1, 4);
  else if (np == 2) FVX_BWDW(1, 2);
  else if (np <= 4) FVX_BWDW(1, 1);
  else if (np <= 8) FVX_BWDW(2, 1);
  else if (np <= 12) FVX_BWDW(3, 1);
  else FVX_BWDW(4, 1);
#undef FVX_BWDW
  red_add(N, li, G, red, s);
}

static void edge_bwdw(UNet& N, int li, const float* s1, const uint16_t* sc, int C, bool swap,
                      int H, int W, RedTable& red, hipStream_t s) {
  const int G = bwdw_slots(N.layers[li], H, W);
  hipLaunchKernelGGL(edge_bwdw_kernel, dim3(G), dim3(256), 0, s, s1, sc, C, swap ? -1 : 1,
                     layer_part(N, li), H, W);
  red_add(N, li, G, red, s);
}

// Backward from N.gy (dLoss/dy, fp32) to weight gradients accumulated in N.g.
static int unet_backward(UNet& N, int H, int W, hipStream_t s) {
  const int L = N.L;
  // output layer
  const Layer& o = N.layers.back();
  const uint16_t* d0 = (L > 1) ? N.dd[0] : N.ee[0];
  take_slots(N, s);
  RedTable red;
  edge_bwdw(N, (int)N.layers.size() - 1, N.gy, d0, N.ch[0], false, H, W, red, s);
  hipLaunchKernelGGL(conv_last_bwd_data_kernel, g2(H, W), dim3(64, 4), 0, s, N.gy, N.w + o.off,
                     N.ch[0], d0, N.gA[0], H, W);
  // decoder levels 0 .. L-2: gA[l] holds the masked gradient into d_l's a2
  for (int l = 0; l <= L - 2; ++l) {
    const int h = H >> l, w = W >> l;
    bwdw_launch(N, layer_index(N, 'd', l), N.h1d[l], N.gA[l], false, h, w, red, s);
    // ga1 = conv^T(ga2) * (h1d > 0) -> gB[l]  (also the skip gradient into e_l)
    conv_launch(N, layer_index(N, 'd', l), true, N.gA[l], N.gB[l], nullptr, N.h1d[l], false, false,
                h, w, s);
    const uint16_t* dnext = (l + 1 == L - 1) ? N.ee[L - 1] : N.dd[l + 1];
    bwdw_launch(N, layer_index(N, 'u', l), dnext, N.gB[l], true, h, w, red, s);
    // gu (fine, C_{l+1} channels) -> gC[l]; up2 backward + relu mask of d_{l+1} -> gA[l+1]
    conv_launch(N, layer_index(N, 'u', l), true, N.gB[l], N.gC[l], nullptr, nullptr, false, false,
                h, w, s);
    const int hc = H >> (l + 1), wc = W >> (l + 1), c = N.ch[l + 1];
    hipLaunchKernelGGL(upbwd_mask_kernel, g1((int64_t)hc * wc * c), dim3(256), 0, s, N.gC[l],
                       dnext, N.gA[l + 1], hc, wc, c);
  }
  // encoder levels L-1 .. 0: gA[l] holds the masked gradient into e_l's a2
  for (int l = L - 1; l >= 0; --l) {
    const int h = H >> l, w = W >> l;
    bwdw_launch(N, layer_index(N, 'b', l), N.h1e[l], N.gA[l], false, h, w, red, s);
    // ga1 = conv^T(ga2) * (h1e > 0) -> gC[l]
    conv_launch(N, layer_index(N, 'b', l), true, N.gA[l], N.gC[l], nullptr, N.h1e[l], false, false,
                h, w, s);
    if (l == 0) {
      edge_bwdw(N, layer_index(N, 'a', 0), N.rin, N.gC[0], N.ch[0], true, h, w, red, s);
      break;
    }
    bwdw_launch(N, layer_index(N, 'a', l), N.xin[l], N.gC[l], false, h, w, red, s);
    // gx = conv^T(ga1) (C_{l-1} channels at level l) -> gA[l] (free now)
    conv_launch(N, layer_index(N, 'a', l), true, N.gC[l], N.gA[l], nullptr, nullptr, false, false,
                h, w, s);
    // gradient into e_{l-1}: (skip grad gB[l-1] + pool^T gx) * (e_{l-1} > 0) -> gA[l-1]
    const int hf = H >> (l - 1), wf = W >> (l - 1), c = N.ch[l - 1];
    hipLaunchKernelGGL(poolbwd_add_mask_kernel, g1((int64_t)hf * wf * c), dim3(256), 0, s,
                       (l - 1 <= L - 2) ? N.gB[l - 1] : nullptr, N.gA[l], N.ee[l - 1],
                       N.gA[l - 1], hf, wf, c);
  }
  red_flush(red, s);
  FVX_LAUNCH_CHECK();
  return kOk;
}

static int repack(UNet& N, hipStream_t s) {
  for (size_t li = 0; li < N.layers.size(); ++li) {
    const Layer& Ly = N.layers[li];
    if (Ly.cin % 16 || Ly.cout % 16) continue;  // edge layers use fp32 weights directly
    hipLaunchKernelGGL(pack_weights_kernel, dim3(64), dim3(256), 0, s, N.w + Ly.off,
                       N.wpk + N.pk_off[li], Ly.cout, Ly.cin, 0);
    hipLaunchKernelGGL(pack_weights_kernel, dim3(64), dim3(256), 0, s, N.w + Ly.off,
                       N.wpkT + N.pk_off[li], Ly.cin, Ly.cout, 1);
  }
  FVX_LAUNCH_CHECK();
  return kOk;
}

}  // namespace fvx

extern "C" {

// channels: nlev entries (each a multiple of 16, <= 64); H, W: the largest
// spatial size the plan will run (divisible by 2^(nlev-1)).
int fvx_unet_create(int nlev, const int* channels, int H, int W, void** out) {
  using namespace fvx;
  FVX_CHECK_ARG(out && channels, "null argument");
  FVX_CHECK_ARG(nlev >= 1 && nlev <= 8, "1..8 levels");
  for (int l = 0; l < nlev; ++l)
    FVX_CHECK_ARG(channels[l] % 16 == 0 && channels[l] >= 16 && channels[l] <= 64,
                  "channels must be multiples of 16 in [16, 64]");
  FVX_CHECK_ARG(H % (1 << (nlev - 1)) == 0 && W % (1 << (nlev - 1)) == 0,
                "H, W must be divisible by 2^(nlev-1)");
  UNet* N = new UNet();
  N->L = nlev;
  for (int l = 0; l < nlev; ++l) N->ch[l] = channels[l];
  N->H = H;
  N->W = W;
  size_t off = 0, pk = 0;
  auto add = [&](int co, int ci) {
    N->layers.push_back({co, ci, off});
    N->pk_off.push_back(pk);
    off += (size_t)9 * co * ci;
    if (co % 16 == 0 && ci % 16 == 0) pk += (size_t)9 * co * ci;
  };
  int cin = 1;
  for (int l = 0; l < nlev; ++l) {
    add(channels[l], cin);
    add(channels[l], channels[l]);
    cin = channels[l];
  }
  for (int l = nlev - 2; l >= 0; --l) {
    add(channels[l], channels[l + 1]);
    add(channels[l], channels[l]);
  }
  add(1, channels[0]);
  N->nweights = off;
  int rc = 0;
  rc |= dev_alloc(*N, &N->w, off);
  rc |= dev_alloc(*N, &N->g, off);
  rc |= dev_alloc(*N, &N->m, off);
  rc |= dev_alloc(*N, &N->v, off);
  rc |= dev_alloc(*N, &N->wpk, pk);
  rc |= dev_alloc(*N, &N->wpkT, pk);
  N->xin.assign(nlev, nullptr);
  N->h1e.assign(nlev, nullptr);
  N->ee.assign(nlev, nullptr);
  N->h1d.assign(nlev, nullptr);
  N->dd.assign(nlev, nullptr);
  N->gA.assign(nlev, nullptr);
  N->gB.assign(nlev, nullptr);
  N->gC.assign(nlev, nullptr);
  for (int l = 0; l < nlev && !rc; ++l) {
    const size_t px = (size_t)(H >> l) * (W >> l);
    const int cmax = std::max(channels[l], l + 1 < nlev ? channels[l + 1] : 0);
    if (l > 0) rc |= dev_alloc(*N, &N->xin[l], px * channels[l - 1]);
    rc |= dev_alloc(*N, &N->h1e[l], px * channels[l]);
    rc |= dev_alloc(*N, &N->ee[l], px * channels[l]);
    rc |= dev_alloc(*N, &N->h1d[l], px * channels[l]);
    rc |= dev_alloc(*N, &N->dd[l], px * channels[l]);
    const int cg = std::max(cmax, l > 0 ? channels[l - 1] : 0);
    rc |= dev_alloc(*N, &N->gA[l], px * cg);
    rc |= dev_alloc(*N, &N->gB[l], px * cg);
    rc |= dev_alloc(*N, &N->gC[l], px * cg);
  }
  const size_t npx = (size_t)H * W;
  rc |= dev_alloc(*N, &N->rin, npx);
  rc |= dev_alloc(*N, &N->yout, npx);
  rc |= dev_alloc(*N, &N->gy, npx);
  rc |= dev_alloc(*N, &N->eref, npx);
  std::vector<size_t> slots;
  for (size_t li = 0; li < N->layers.size(); ++li) {
    const Layer& Ly = N->layers[li];
    const int k = (int)li, l = k < 2 * nlev ? k / 2 : (k == (int)N->layers.size() - 1 ? 0 : nlev - 2 - (k - 2 * nlev) / 2);
    slots.push_back((size_t)bwdw_slots(Ly, H >> l, W >> l) * 9 * Ly.cout * Ly.cin);
    if (slots[li] > slots[N->widest]) N->widest = (int)li;
  }
  for (size_t li = 0; li < slots.size(); ++li) {
    N->part_off.push_back(N->rest_elems);
    if ((int)li != N->widest) N->rest_elems += slots[li];
  }
  rc |= dev_alloc(*N, &N->part, slots[N->widest]);
  rc |= dev_alloc(*N, &N->rms_part, 4096);
  rc |= dev_alloc(*N, &N->scal, 4);
  rc |= dev_alloc(*N, &N->loss, 1);
  if (!rc) {
    const int big = 160 * 1024;
#define FVX_BWDW_LDS(PW, RS)                                                          \
  (void)hipFuncSetAttribute((const void*)conv_bwdw_mfma_kernel<PW, RS, true>,         \
                            hipFuncAttributeMaxDynamicSharedMemorySize, big);         \
  (void)hipFuncSetAttribute((const void*)conv_bwdw_mfma_kernel<PW, RS, false>,        \
                            hipFuncAttributeMaxDynamicSharedMemorySize, big)
    FVX_BWDW_LDS(1, 4);
    FVX_BWDW_LDS(1, 2);
    FVX_BWDW_LDS(1, 1);
    FVX_BWDW_LDS(2, 1);
    FVX_BWDW_LDS(3, 1);
    FVX_BWDW_LDS(4, 1);
#undef FVX_BWDW_LDS
    hipError_t e = hipMemset(N->g, 0, off * sizeof(float));
    if (e == hipSuccess) e = hipMemset(N->m, 0, off * sizeof(float));
    if (e == hipSuccess) e = hipMemset(N->v, 0, off * sizeof(float));
    if (e != hipSuccess) rc = kHipError;
  }
  if (rc) {
    for (void* p : N->allocs) (void)hipFree(p);
    delete N;
    if (rc != kInvalidArgument) set_error("allocation failed for the U-Net plan");
    return rc == kInvalidArgument ? rc : kHipError;
  }
  *out = N;
  return kOk;
}

int fvx_unet_destroy(void* net) {
  using namespace fvx;
  if (!net) return kOk;
  UNet* N = (UNet*)net;
  (void)hipDeviceSynchronize();
  for (void* p : N->allocs) (void)hipFree(p);
  delete N;
  return kOk;
}

// Number of fp32 weights (all layers, layout [9][Cout][Cin] per layer in the
// order e0a e0b .. e{L-1}b, u{L-2} d{L-2} .. u0 d0, out).
int64_t fvx_unet_num_weights(void* net) { return net ? (int64_t)((fvx::UNet*)net)->nweights : -1; }

// Copy fp32 weights in (device pointer) or out; resets Adam state on "in".
int fvx_unet_weights(void* net, float* w, int direction, void* stream) {
  using namespace fvx;
  FVX_CHECK_ARG(net && w, "null argument");
  UNet* N = (UNet*)net;
  hipStream_t s = (hipStream_t)stream;
  if (direction == 0) {
    FVX_HIP(hipMemcpyAsync(N->w, w, N->nweights * sizeof(float), hipMemcpyDeviceToDevice, s));
    FVX_HIP(hipMemsetAsync(N->m, 0, N->nweights * sizeof(float), s));
    FVX_HIP(hipMemsetAsync(N->v, 0, N->nweights * sizeof(float), s));
    FVX_HIP(hipMemsetAsync(N->g, 0, N->nweights * sizeof(float), s));
    N->adam_t = 0;
    return repack(*N, s);
  }
  FVX_HIP(hipMemcpyAsync(w, N->w, N->nweights * sizeof(float), hipMemcpyDeviceToDevice, s));
  return kOk;
}

// Raw forward on an fp32 (H, W) input already in the network's units:
// y = net(x).  H, W <= the plan's size and divisible by 2^(L-1).
int fvx_unet_forward_raw(void* net, const float* x, float* y, int H, int W, void* stream) {
  using namespace fvx;
  FVX_CHECK_ARG(net && x && y, "null argument");
  UNet* N = (UNet*)net;
  FVX_CHECK_ARG(H <= N->H && W <= N->W && H * W <= N->H * N->W, "input larger than the plan");
  FVX_CHECK_ARG(H % (1 << (N->L - 1)) == 0 && W % (1 << (N->L - 1)) == 0, "size not divisible");
  hipStream_t s = (hipStream_t)stream;
  FVX_HIP(hipMemcpyAsync(N->rin, x, (size_t)H * W * sizeof(float), hipMemcpyDeviceToDevice, s));
  int rc = unet_forward(*N, H, W, s);
  if (rc) return rc;
  FVX_HIP(hipMemcpyAsync(y, N->yout, (size_t)H * W * sizeof(float), hipMemcpyDeviceToDevice, s));
  return kOk;
}

// Weight gradients of sum(gy * net(x)) accumulated into the plan's gradient
// buffer (read with fvx_unet_grads); for tests and training.
int fvx_unet_backward_raw(void* net, const float* x, const float* gy, int H, int W,
                          void* stream) {
  using namespace fvx;
  FVX_CHECK_ARG(net && x && gy, "null argument");
  UNet* N = (UNet*)net;
  FVX_CHECK_ARG(H <= N->H && W <= N->W, "input larger than the plan");
  hipStream_t s = (hipStream_t)stream;
  FVX_HIP(hipMemcpyAsync(N->rin, x, (size_t)H * W * sizeof(float), hipMemcpyDeviceToDevice, s));
  int rc = unet_forward(*N, H, W, s);
  if (rc) return rc;
  FVX_HIP(hipMemcpyAsync(N->gy, gy, (size_t)H * W * sizeof(float), hipMemcpyDeviceToDevice, s));
  return unet_backward(*N, H, W, s);
}

int fvx_unet_grads(void* net, float* g, int zero_after, void* stream) {
  using namespace fvx;
  FVX_CHECK_ARG(net && g, "null argument");
  UNet* N = (UNet*)net;
  hipStream_t s = (hipStream_t)stream;
  FVX_HIP(hipMemcpyAsync(g, N->g, N->nweights * sizeof(float), hipMemcpyDeviceToDevice, s));
  if (zero_after) FVX_HIP(hipMemsetAsync(N->g, 0, N->nweights * sizeof(float), s));
  return kOk;
}

// One training step on a batch of B pairs (x_b, e_b), each (H, W) fp32 in the
// network's units: loss = mean_b mean_p (net(x_b) - e_b)^2; Adam update.
// Returns the batch loss in *loss_out (synchronises the stream).
int fvx_unet_train_step(void* net, const float* xb, const float* eb, int B, int H, int W,
                        double lr, double* loss_out, void* stream) {
  using namespace fvx;
  FVX_CHECK_ARG(net && xb && eb && B >= 1, "bad arguments");
  UNet* N = (UNet*)net;
  FVX_CHECK_ARG(H <= N->H && W <= N->W, "batch item larger than the plan");
  hipStream_t s = (hipStream_t)stream;
  FVX_HIP(hipMemsetAsync(N->loss, 0, sizeof(double), s));
  const size_t npx = (size_t)H * W;
  for (int b = 0; b < B; ++b) {
    FVX_HIP(hipMemcpyAsync(N->rin, xb + b * npx, npx * sizeof(float), hipMemcpyDeviceToDevice, s));
    int rc = unet_forward(*N, H, W, s);
    if (rc) return rc;
    hipLaunchKernelGGL(mse_grad_kernel, g1((int64_t)npx), dim3(256), 0, s, N->yout, eb + b * npx,
                       N->gy, (int64_t)npx, N->loss);
    rc = unet_backward(*N, H, W, s);
    if (rc) return rc;
  }
  N->adam_t += 1;
  const float b1 = 0.9f, b2 = 0.999f;
  const float bc1 = 1.f - std::pow(b1, (float)N->adam_t), bc2 = 1.f - std::pow(b2, (float)N->adam_t);
  hipLaunchKernelGGL(adam_kernel, g1((int64_t)N->nweights), dim3(256), 0, s, N->w, N->g, N->m,
                     N->v, (int64_t)N->nweights, (float)lr, b1, b2, 1e-8f, bc1, bc2, 1.0f / B);
  int rc = repack(*N, s);
  if (rc) return rc;
  double l = 0.0;
  FVX_HIP(hipMemcpyAsync(&l, N->loss, sizeof(double), hipMemcpyDeviceToHost, s));
  FVX_HIP(hipStreamSynchronize(s));
  if (loss_out) *loss_out = l / B;
  return kOk;
}

}  // extern "C"

// Preconditioner application for PCG: z = out_scale * rms(r) * net(r / rms(r)) * mask.
namespace fvx {
template <typename T>
int unet_apply(void* net, const T* r, int64_t ld_r, T* z, int64_t ld_z, int H, int W,
               double out_scale, const uint8_t* mask, hipStream_t s, const int* guard) {
  UNet* N = (UNet*)net;
  N->guard = guard;
  FVX_CHECK_ARG(H <= N->H && W <= N->W, "field larger than the network plan");
  FVX_CHECK_ARG(H % (1 << (N->L - 1)) == 0 && W % (1 << (N->L - 1)) == 0,
                "field size not divisible by 2^(levels-1)");
  const int nb = 256;
  hipLaunchKernelGGL(rms_kernel<T>, dim3(nb), dim3(256), 0, s, r, ld_r, H, W, N->rms_part,
                     N->guard);
  hipLaunchKernelGGL(rms_finish_kernel, dim3(1), dim3(256), 0, s, N->rms_part, nb,
                     (int64_t)H * W, N->scal, out_scale, N->guard);
  hipLaunchKernelGGL(scale_in_kernel<T>, g2(H, W), dim3(64, 4), 0, s, r, ld_r, H, W, N->scal,
                     N->rin, N->guard);
  int rc = unet_forward(*N, H, W, s, false);
  if (rc) return rc;
  // Output conv with the rescaling and mask fused.
  hipLaunchKernelGGL((conv_last_kernel<T>), g2(H, W), dim3(64, 4), 0, s,
                     (N->L > 1) ? N->dd[0] : N->ee[0], N->w + N->layers.back().off, N->ch[0], z,
                     ld_z, H, W, N->scal + 1, mask, N->guard);
  N->guard = nullptr;
  FVX_LAUNCH_CHECK();
  return kOk;
}
template int unet_apply<float>(void*, const float*, int64_t, float*, int64_t, int, int, double,
                               const uint8_t*, hipStream_t, const int*);
template int unet_apply<double>(void*, const double*, int64_t, double*, int64_t, int, int, double,
                                const uint8_t*, hipStream_t, const int*);
}  // namespace fvx

// Standalone 3x3 conv (bf16 HWC in/out, fp32 weights [9][Cout][Cin], Cin and
// Cout multiples of 16 <= 64), optionally reading x through nearest
// upsampling and applying ReLU.  ``scratch`` holds >= 9*Cout*Cin bf16.
extern "C" int fvx_conv3x3_bf16(const uint16_t* x, int Cin, const float* w, int Cout,
                                uint16_t* out, int H, int W, int ups, int relu, uint16_t* scratch,
                                void* stream) {
  using namespace fvx;
  FVX_CHECK_ARG(x && w && out && scratch, "null argument");
  FVX_CHECK_ARG(Cin % 16 == 0 && Cout % 16 == 0 && Cin <= 64 && Cout <= 64 && Cin > 0 && Cout > 0,
                "channels must be multiples of 16 in [16, 64]");
  FVX_CHECK_ARG(!ups || (H % 2 == 0 && W % 2 == 0), "upsampling needs even H, W");
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(pack_weights_kernel, dim3(64), dim3(256), 0, s, w, scratch, Cout, Cin, 0);
  UNet N;
  N.layers.push_back({Cout, Cin, 0});
  N.pk_off.push_back(0);
  N.wpk = scratch;
  N.wpkT = scratch;
  conv_launch(N, 0, false, x, out, nullptr, nullptr, relu != 0, ups != 0, H, W, s);
  FVX_LAUNCH_CHECK();
  return kOk;
}

extern "C" int fvx_unet_apply_f32(void* net, const float* r, int64_t ld_r, float* z, int64_t ld_z,
                                  int H, int W, double out_scale, const uint8_t* mask,
                                  void* stream) {
  if (!net || !r || !z) {
    fvx::set_error("null argument");
    return fvx::kInvalidArgument;
  }
  return fvx::unet_apply<float>(net, r, ld_r, z, ld_z, H, W, out_scale, mask, (hipStream_t)stream,
                                nullptr);
}
