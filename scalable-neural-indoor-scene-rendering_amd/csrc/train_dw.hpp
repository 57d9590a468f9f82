// Weight-gradient reduction shared by the FP32 training kernels: dW += D^T A and db += sum D over a range
// of stored 32-record blocks (train_mma.hpp's row layout), the records as the K dimension.
#pragma once

#include "train_mma.hpp"

namespace snisr {

// One wavefront's share of a layer: NA output blocks from ob0 and NB input blocks from ib0 over the record
// blocks j0, j0 + dj, ... < j1.  A lane of an operand is a feature and its k slots are records, so both
// operands come straight from memory in 1 KB loads (no LDS, no barriers), the next half block's loads in
// flight while the current one is split into its BF16 parts and multiplied.
// OW / IW: row widths, OUTL / INL: real outputs and inputs.  ONCE: no other
// wavefront reads these blocks, so the loads are non-temporal (1.56 GB of the 530k-sample reflection step: 360 -> 265
// us with the rows stored so too; blocks that two wavefronts share are 7% slower that way: 2283 -> 2450 us at width 128).
// With `red` (NA NB 1024 floats of LDS) the workgroup's wavefronts hold the same blocks: they are added there
// first and only the sums go out.
// flip: the sums are formed with D's sign changed, and changed back at the end.  BF16 matrix products round their
// sums towards minus infinity; half of the wavefronts or splits that add to one gradient are flipped, so that the
// errors cancel.  Weight gradients of 530k samples, relative to 64 bits: FP32 products 1.07e-6, these without the flip
// 1.20e-6 with a mean error of -1.6 deviations, 5.7e-7 with it (2% of this kernel's time).
template <int OW, int IW, int OUTL, int INL, int NA, int NB, bool ONCE>
__device__ __forceinline__ void dw_wave(const float* __restrict__ D, const float* __restrict__ A, int64_t j0, int64_t j1,
                                        int64_t dj, int ob0, int ib0, float* __restrict__ G, bool flip, float* red = nullptr) {
  const uint32_t sign = flip ? 0x80000000u : 0u;
  auto signed_of = [&](float v) { return __uint_as_float(__float_as_uint(v) ^ sign); };
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  f32x16 acc[NA][NB];
  float db[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    db[i] = 0.0f;
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x16{};
  }
  // values of k-chunk kc (records 16 kc .. +15) of block b of a W-wide row: two pieces of four records
  float nd[NA][8], na[NB][8];
  auto load = [&](const float* rows, int64_t blk, int W, int b, int kc, float (&v)[8]) {
    const int w = W - 32 * b < 32 ? W - 32 * b : 32;
    const float* p = rows + blk * 32 * W + 1024 * b + 4 * c;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      f32x4 t = {0.0f, 0.0f, 0.0f, 0.0f};
      if (c < w) {
        const f32x4* from = reinterpret_cast<const f32x4*>(p + 4 * w * (4 * kc + 2 * u + h));
        t = ONCE ? __builtin_nontemporal_load(from) : *from;
      }
      v[4 * u] = t.x;
      v[4 * u + 1] = t.y;
      v[4 * u + 2] = t.z;
      v[4 * u + 3] = t.w;
    }
  };
  auto fetch = [&](int64_t blk, int kc) {
#pragma unroll
    for (int i = 0; i < NA; ++i) load(D, blk, OW, ob0 + i, kc, nd[i]);
#pragma unroll
    for (int j = 0; j < NB; ++j) load(A, blk, IW, ib0 + j, kc, na[j]);
  };
  if (j0 < j1) fetch(j0, 0);
#pragma unroll 1
  for (int64_t blk = j0; blk < j1; blk += dj) {
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      Split8 a[NA], b[NB];
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        float sd[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) sd[e] = signed_of(nd[i][e]);
        a[i] = split8(sd);
        db[i] += ((nd[i][0] + nd[i][1]) + (nd[i][2] + nd[i][3])) + ((nd[i][4] + nd[i][5]) + (nd[i][6] + nd[i][7]));
      }
#pragma unroll
      for (int j = 0; j < NB; ++j) b[j] = split8(na[j]);
      if (kc == 0) fetch(blk, 1);
      else if (blk + dj < j1) fetch(blk + dj, 0);
      mma_split<NA, NB>(a, b, acc);
    }
  }
#pragma unroll
  for (int i = 0; i < NA; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = signed_of(acc[i][j][r]);
  const int wv = threadIdx.x >> 6;
  if (red) {
    for (int w = 1; w < 4; ++w) {  // wavefront w hands its sums to wavefront 0
      __syncthreads();
      if (wv == w) {
#pragma unroll
        for (int i = 0; i < NA; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) red[((i * NB + j) * 16 + r) * 64 + lane] = acc[i][j][r];
      }
      __syncthreads();
      if (wv == 0) {
#pragma unroll
        for (int i = 0; i < NA; ++i)
#pragma unroll
          for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] += red[((i * NB + j) * 16 + r) * 64 + lane];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NA; ++i) {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      if (red && wv) break;
      const int in = 32 * (ib0 + j) + c;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int o = 32 * (ob0 + i) + 8 * (r / 4) + 4 * h + (r % 4);
        if (o < OUTL && in < INL && acc[i][j][r] != 0.0f) atomicAdd(&G[(int64_t)o * INL + in], acc[i][j][r]);
      }
    }
    const float s = db[i] + __shfl_xor(db[i], 32);
    const int o = 32 * (ob0 + i) + c;
    if (ib0 == 0 && h == 0 && o < OUTL && s != 0.0f) atomicAdd(&G[(int64_t)OUTL * INL + o], s);
  }
}

// dW_l[o][i] += sum_j D_l[j][o] A_l[j][i] and db_l[o] += sum_j D_l[j][o] over the record blocks [j0, j1) of a
// four-wavefront workgroup.  A layer of at most 2 x 2 blocks gives every wavefront all of them over every
// fourth record block (red: 4096 floats of LDS); a larger one gives each wavefront a part of the blocks over all records.
template <int OW, int IW, int OUTL, int INL>
__device__ __forceinline__ void dw_layer(const float* __restrict__ D, const float* __restrict__ A, int64_t j0, int64_t j1,
                                         float* __restrict__ G, float* red) {
  constexpr int NOB = (OUTL + 31) / 32, NIB = (INL + 31) / 32;
  const int wv = threadIdx.x >> 6;
  const bool odd = blockIdx.x & 1;  // of the splits of a layer
  if constexpr (NOB <= 2 && NIB <= 2) {
    dw_wave<OW, IW, OUTL, INL, NOB, NIB, true>(D, A, j0 + wv, j1, 4, 0, 0, G, wv & 1, red);
  } else if constexpr (NOB == 4 && NIB == 4) {
    dw_wave<OW, IW, OUTL, INL, 2, 2, false>(D, A, j0, j1, 1, 2 * (wv >> 1), 2 * (wv & 1), G, odd);
  } else if constexpr (NOB == 4 && NIB == 2) {
    dw_wave<OW, IW, OUTL, INL, 2, 1, false>(D, A, j0, j1, 1, 2 * (wv >> 1), wv & 1, G, odd);
  } else {
    static_assert(NOB == 1 && NIB == 4, "layer shapes of the training MLPs");
    dw_wave<OW, IW, OUTL, INL, 1, 2, false>(D, A, j0 + (wv >> 1), j1, 2, 0, 2 * (wv & 1), G, (wv >> 1) != odd);
  }
}

}  // namespace snisr
