// Matrix-product building blocks of the FP32 training MLPs (the feature-scene training chain and the
// positional-encoding MLP): FP32 operands as sums of 16-bit parts, the packing of the weights, their staging
// through LDS and the product of one layer.
//
// A layer's product W x runs on v_mfma_f32_32x32x16_f16 with both operands as two FP16 parts: the operand is
// scaled by a power of two so that its largest magnitude (of the layer's weights; of the activation column)
// lies in [2^14, 2^15), hi = the scaled value rounded to FP16, lo = the rounded remainder, and
// W x = hi hi + hi lo + lo hi, accumulated in FP32 and scaled back exactly.  hi + lo keeps 22 bits and lo lo
// is below 2^-22, both of random sign; a value 2^-16 of its column's largest still keeps them.  The three
// products sum 16 terms per rounding where v_mfma_f32_32x32x2_f32 sums two, and the errors against 64 bits
// are those of the FP32 products or smaller (relative, FP32 products | these: parameter gradients of the
// 530k-sample reflection step 9.0e-6 | 4.7e-6, of the diffuse step 3.1e-5 | 3.1e-5, feature gradients of the
// 131k-ray step 9.1e-3 | 9.1e-3, where the march's positions set them).  An infinite operand gives NaN (its
// remainder is inf - inf).
//
// Against FP32 products with weights read from L2 by every wavefront (3.04M records at width 128; 530k samples
// of the reflection MLP; us): forward 2502 -> 1146; 305 -> 108, backward 6654 -> 4240; 572 -> 301.  With
// three BF16 parts and six products the forward took 2160; 212: under matrix load the card holds about half
// of its nominal rate, so the products themselves are what is worth saving.
//
// Sums over records (the weight gradients) have no common scale: their operands are split into three BF16
// parts, which keep the range and all 24 bits of FP32, and multiplied as six products (what is left out is
// below 2^-26).
#pragma once

#include "mfma_ops.hpp"
#include "snisr_device.hpp"

namespace snisr {

// One wavefront takes 32 records of one tile as the 32 columns, so every layer is W (out x in) times a
// 32-column block of activations.  Lane layouts of v_mfma_f32_32x32x16 (h = lane / 32, c = lane % 32):
//   A:  lane holds A[row c][k slots 8h .. 8h+7]      B:  lane holds B[k slots 8h .. 8h+7][column c]
//   D:  lane holds rows 8(r/4) + 4h + (r%4), r = 0..15, of column c
// Register s of a lane's activations holds row tr_row(s, h): the order in which the D blocks of a layer
// come out.  K slot e of half h in k-chunk kc is row tr_row(8 kc + e, h), so the B operand of a chunk is
// registers 8 kc .. 8 kc + 7 of the previous layer's output and activations never leave registers.
// Layer 0's inputs (features, then the view encoding) follow the same row order.
__host__ __device__ constexpr int tr_row(int s, int h) { return 32 * (s / 16) + 8 * ((s % 16) / 4) + 4 * h + (s % 4); }
// registers of layer 0's inputs: whole 8-row groups
__host__ __device__ constexpr int tr_ns0(int in0) { return 16 * (in0 / 32) + 4 * ((in0 % 32 + 7) / 8); }

// Packed weights: a fragment is 32 output rows x 16 k, its two parts of 64 lanes x 16 bytes; the fragments
// of a layer are ordered k-chunk by k-chunk, output block by output block, and padded to whole groups of
// kChunkFrags, the unit that is staged through LDS.  Order: the forward layers 0 .. L-1, the transposed
// layers L-1 .. 0, i.e. the order in which the kernels read them; then the biases (32 floats per output
// block, in the D layout) and one factor per layer, the inverse of its weights' scale.
constexpr int kPartBytes = 1024, kFragBytes = 2 * kPartBytes, kChunkFrags = 8, kChunkBytes = kChunkFrags * kFragBytes;
__host__ __device__ constexpr int tr_nob(int wd, int L, int l) { return l == L - 1 ? 1 : wd / 32; }
__host__ __device__ constexpr int tr_nkf(int in0, int wd, int l) { return l == 0 ? (tr_ns0(in0) + 7) / 8 : wd / 16; }
__host__ __device__ constexpr int tr_nib(int wd, int l) { return l == 0 ? 1 : wd / 32; }
__host__ __device__ constexpr int tr_nkb(int wd, int L, int l, int nout) { return l == L - 1 ? (nout + 15) / 16 : wd / 16; }
__host__ __device__ constexpr int tr_chunks(int frags) { return (frags + kChunkFrags - 1) / kChunkFrags; }
// chunks before forward layer l (l = L: all forward chunks)
__host__ __device__ constexpr int tr_fwd_chunk(int in0, int wd, int L, int l) {
  int n = 0;
  for (int m = 0; m < l; ++m) n += tr_chunks(tr_nkf(in0, wd, m) * tr_nob(wd, L, m));
  return n;
}
// chunks before transposed layer l, which follows layer l + 1 (l = -1: all chunks)
__host__ __device__ constexpr int tr_bwd_chunk(int in0, int wd, int L, int l, int nout) {
  int n = tr_fwd_chunk(in0, wd, L, L);
  for (int m = L - 1; m > l; --m) n += tr_chunks(tr_nkb(wd, L, m, nout) * tr_nib(wd, m));
  return n;
}
// float offset of layer l's biases in the packed block, and the block's floats
__host__ __device__ constexpr int64_t tr_bias_off(int in0, int wd, int L, int l, int nout) {
  int64_t o = (int64_t)tr_bwd_chunk(in0, wd, L, -1, nout) * (kChunkBytes / 4);
  for (int m = 0; m < l; ++m) o += 32 * tr_nob(wd, L, m);
  return o;
}
// float offset of the layers' factors, and the floats of a packed block
__host__ __device__ constexpr int64_t tr_scale_off(int in0, int wd, int L, int nout) { return tr_bias_off(in0, wd, L, L, nout); }
__host__ __device__ constexpr int64_t tr_stride(int in0, int wd, int L, int nout) {
  return (tr_scale_off(in0, wd, L, nout) + L + 63) / 64 * 64;
}

// power of two that brings a largest magnitude into [2^14, 2^15), and its inverse (magnitudes below 2^-112
// count as 2^-112)
__device__ __forceinline__ void range_scale(float largest, float& scale, float& inverse) {
  uint32_t e = __float_as_uint(largest) >> 23;
  e = e < 15u ? 15u : (e > 254u ? 254u : e);
  scale = __uint_as_float((268u - e) << 23);
  inverse = __uint_as_float((e - 14u) << 23);
}

// hi + lo of eight scaled values
struct Pair8 {
  f16x8 hi, lo;
};
__device__ __forceinline__ Pair8 pair8(const float* v, float scale) {
  Pair8 s;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const _Float16 h = (_Float16)(v[e] * scale);
    s.hi[e] = h;
    s.lo[e] = (_Float16)__builtin_fmaf(v[e], scale, -(float)h);
  }
  return s;
}

// x = hi + mid + lo of eight values, each part rounded to nearest BF16
struct Split8 {
  bf16x8 p[3];
};
__device__ __forceinline__ Split8 split8(const float* v) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  uint32_t w[3][4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float a = v[2 * q], b = v[2 * q + 1];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
      w[i][q] = u;
      if (i < 2) {
        a = a - __uint_as_float(u << 16);
        b = b - __uint_as_float(u & 0xffff0000u);
      }
    }
  }
  Split8 s;
#pragma unroll
  for (int i = 0; i < 3; ++i) s.p[i] = __builtin_bit_cast(bf16x8, make_uint4(w[i][0], w[i][1], w[i][2], w[i][3]));
  return s;
}

// acc[i][j] += a[i] b[j] for NA x NB blocks, small products first; consecutive products are independent
template <int NA, int NB>
__device__ __forceinline__ void mma_split(const Split8 (&a)[NA], const Split8 (&b)[NB], f32x16 (&acc)[NA][NB]) {
  constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
  for (int q = 0; q < 6; ++q)
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i].p[pa[q]], b[j].p[pb[q]], acc[i][j], 0, 0, 0);
}

namespace {
constexpr int kPackThreads = 512;
// One workgroup per layer and tile: the largest magnitude of the layer's weights, then its forward and
// transposed fragments, its biases and its factor (mlp_params layout: per layer W[out][in], then b[out]; the
// last layer has nout <= 32 rows).  in_of(row): the input at row `row` of layer 0's products.
template <class InOf>
__device__ __forceinline__ void pack_train_layer(const float* __restrict__ P, float* __restrict__ block, int in0, int wd,
                                                 int L, int l, int nout, InOf in_of) {
  __shared__ float wmax[kPackThreads / 64];
  for (int m = 0; m < l; ++m) P += (int64_t)((m == 0 ? in0 : wd) + 1) * wd;
  const int in = l == 0 ? in0 : wd, out = l == L - 1 ? nout : wd;
  float mx = 0.0f;
  for (int q = threadIdx.x; q < in * out; q += kPackThreads) mx = fmaxf(mx, fabsf(P[q]));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = mx;
  __syncthreads();
  for (int w = 0; w < kPackThreads / 64; ++w) mx = fmaxf(mx, wmax[w]);
  float scale, inverse;
  range_scale(mx, scale, inverse);
  if (threadIdx.x == 0) block[tr_scale_off(in0, wd, L, nout) + l] = inverse;
  const int nob = tr_nob(wd, L, l);
  float* bias = block + tr_bias_off(in0, wd, L, l, nout);
  for (int q = threadIdx.x; q < 32 * nob; q += kPackThreads) {
    const int o = 32 * (q / 32) + 8 * (q % 16 / 4) + 4 * (q / 16 % 2) + q % 4;
    bias[q] = o < out ? P[(int64_t)out * in + o] : 0.0f;
  }
  for (int bwd = 0; bwd < 2; ++bwd) {
    const int nblk = bwd ? tr_nib(wd, l) : nob, nk = bwd ? tr_nkb(wd, L, l, nout) : tr_nkf(in0, wd, l);
    const int c0 = bwd ? tr_bwd_chunk(in0, wd, L, l, nout) : tr_fwd_chunk(in0, wd, L, l);
    uint8_t* to = reinterpret_cast<uint8_t*>(block) + (int64_t)c0 * kChunkBytes;
    const int slots = tr_chunks(nk * nblk) * kChunkFrags * 64;
    for (int q = threadIdx.x; q < slots; q += kPackThreads) {
      const int f = q / 64, lane = q % 64, h = lane / 32, kc = f / nblk, row = 32 * (f % nblk) + lane % 32;
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int k = tr_row(8 * kc + e, h);
        int o = bwd ? k : row, i = bwd ? row : k;
        if (l == 0) i = in_of(i);
        v[e] = kc < nk && o < out && i < in ? P[(int64_t)o * in + i] : 0.0f;
      }
      const Pair8 s = pair8(v, scale);
      *reinterpret_cast<f16x8*>(to + (int64_t)f * kFragBytes + lane * 16) = s.hi;
      *reinterpret_cast<f16x8*>(to + (int64_t)f * kFragBytes + kPartBytes + lane * 16) = s.lo;
    }
  }
}
}  // namespace

// The weight stream of a 256-thread workgroup: chunks of kChunkFrags fragments go from global memory
// through registers into one of two LDS buffers, the next chunk's loads in flight while the current one is
// used.  Without the staging every wavefront would read every fragment from L2 (3 KB per six products).
// All wavefronts of the workgroup call start() and the same number of step()s.
struct FragStream {
  static constexpr int kThreads = 256;
  static_assert(kChunkBytes == 4 * 16 * kThreads, "four 16-byte pieces per thread and chunk");
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  u32x4 r0, r1, r2, r3;
  const u32x4* src;
  u32x4* lds;  // 2 * kChunkBytes
  int left;    // chunks after the one being fetched
  int cur;
  // unconditional: past the last chunk it reads that chunk again (a conditional load would be merged with
  // the registers' old values through memory)
  __device__ __forceinline__ void fetch() {
    r0 = src[0];
    r1 = src[kThreads];
    r2 = src[2 * kThreads];
    r3 = src[3 * kThreads];
    src += left > 0 ? kChunkBytes / 16 : 0;
    --left;
  }
  __device__ __forceinline__ void start(const float* packed, uint8_t* buf, int chunks) {
    src = reinterpret_cast<const u32x4*>(packed) + threadIdx.x;
    lds = reinterpret_cast<u32x4*>(buf);
    left = chunks - 1;
    cur = 1;
    fetch();
  }
  // the next chunk, in LDS; the buffer it replaces was read before the previous step's barrier
  __device__ __forceinline__ const uint8_t* step() {
    cur ^= 1;
    u32x4* b = lds + cur * (kChunkBytes / 16);
    b[threadIdx.x] = r0;
    b[threadIdx.x + kThreads] = r1;
    b[threadIdx.x + 2 * kThreads] = r2;
    b[threadIdx.x + 3 * kThreads] = r3;
    __syncthreads();
    fetch();
    return reinterpret_cast<const uint8_t*>(b);
  }
};

// largest magnitude of this lane's column: N values here, the others in the lane of the other half
template <int N>
__device__ __forceinline__ float column_max(const float* x) {
  float m = 0.0f;
#pragma unroll
  for (int r = 0; r < N; ++r) m = fmaxf(m, fabsf(x[r]));
  float lo, hi;
  swap_halves(m, lo, hi);
  return fmaxf(lo, hi);
}

// out(i, y) for register i of the NOB output blocks, y = (the layer's fragments times x) + bias; x: registers
// s (row tr_row(s, h)) over NK k-chunks, at least 8 NK values; weight_inv: the layer's factor; bias: NOB
// blocks of 32 floats, or NULL.  All output blocks advance together, so x is split once and consecutive
// products are independent; the small products come first in a k-chunk.
template <int NK, int NOB, class Out>
__device__ __forceinline__ void stream_layer(FragStream& fs, const float* x, int lane, float weight_inv,
                                             const float* __restrict__ bias, Out out) {
  static_assert(kChunkFrags % NOB == 0, "whole k-chunks per staged chunk");
  constexpr int KPC = kChunkFrags / NOB;
  float scale, inv;
  range_scale(column_max<8 * NK>(x), scale, inv);
  inv *= weight_inv;
  f32x16 acc[NOB];
#pragma unroll
  for (int ob = 0; ob < NOB; ++ob) acc[ob] = f32x16{};
#pragma unroll
  for (int k0 = 0; k0 < NK; k0 += KPC) {
    const uint8_t* A = fs.step();
#pragma unroll
    for (int k = 0; k < KPC; ++k)
      if (k0 + k < NK) {
        f16x8 hi[NOB], lo[NOB];
        const Pair8 b = pair8(x + 8 * (k0 + k), scale);
#pragma unroll
        for (int ob = 0; ob < NOB; ++ob) {
          hi[ob] = load_frag<f16x8>(A + (k * NOB + ob) * kFragBytes + lane * 16);
          lo[ob] = load_frag<f16x8>(A + (k * NOB + ob) * kFragBytes + kPartBytes + lane * 16);
        }
#pragma unroll
        for (int ob = 0; ob < NOB; ++ob) acc[ob] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo[ob], b.hi, acc[ob], 0, 0, 0);
#pragma unroll
        for (int ob = 0; ob < NOB; ++ob) acc[ob] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi[ob], b.lo, acc[ob], 0, 0, 0);
#pragma unroll
        for (int ob = 0; ob < NOB; ++ob) acc[ob] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi[ob], b.hi, acc[ob], 0, 0, 0);
      }
  }
#pragma unroll
  for (int ob = 0; ob < NOB; ++ob) {
    f32x16 b = f32x16{};
    if (bias) b = bias_block(bias, ob, lane >> 5);
#pragma unroll
    for (int r = 0; r < 16; ++r) out(16 * ob + r, bias ? __builtin_fmaf(acc[ob][r], inv, b[r]) : acc[ob][r] * inv);
  }
}

__device__ __forceinline__ void store4(float* p, const float* v) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}

// ---------------------------------------------------------------------------- stored rows
// The weight gradients reduce over records, so their operands are read with the records along K: the
// rows of a 32-record block are stored as pieces of four records of one feature (16 bytes), feature block
// by feature block: block b of 32 features (the last one may hold fewer, a multiple of 4) starts at
// 1024 b floats and holds piece (record quad q, feature f) at 4 (q w + f % 32), w its width.  The 64 lanes
// of a load then read 1 KB in a row as an MFMA operand (lane = feature), and the writer's stores cover
// whole lines.

// exchange within groups of four lanes: lane i gives value j to lane j, which keeps it as value i
__device__ __forceinline__ void quad_transpose(float (&v)[4]) {
  const bool o1 = threadIdx.x & 1, o2 = threadIdx.x & 2;
  auto swap = [&](float& lo, float& hi, bool upper, auto dpp) {
    const float got = __int_as_float(dpp(__float_as_int(upper ? lo : hi)));
    lo = upper ? got : lo;
    hi = upper ? hi : got;
  };
  auto x1 = [](int a) { return __builtin_amdgcn_mov_dpp(a, 0xB1, 0xf, 0xf, true); };  // lane ^ 1
  auto x2 = [](int a) { return __builtin_amdgcn_mov_dpp(a, 0x4E, 0xf, 0xf, true); };  // lane ^ 2
  swap(v[0], v[1], o1, x1);
  swap(v[2], v[3], o1, x1);
  swap(v[0], v[2], o2, x2);
  swap(v[1], v[3], o2, x2);
}

// stores registers 4g .. 4g+3 (rows 8(g%4) + 4h .. +3 of feature block g / 4) of this wavefront's 32 records
// for NG groups of a layer of width W (a multiple of 8, or 4: lane half 0 only); called by whole wavefronts.
// The rows are read once, by another kernel and long after: non-temporal stores keep them from displacing the weights
// and features (backward of 3.04M records at width 128: 4420 -> 4240 us).
typedef float f32x4 __attribute__((ext_vector_type(4)));
template <int W, int NG>
__device__ __forceinline__ void store_rows(float* __restrict__ block, const float* x, int lane) {
  const int c = lane & 31, h = lane >> 5, q = c >> 2, i = c & 3;
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    float v[4] = {x[4 * g], x[4 * g + 1], x[4 * g + 2], x[4 * g + 3]};
    quad_transpose(v);
    const int b = g / 4, w = W - 32 * b < 32 ? W - 32 * b : 32;
    float* to = block + 1024 * b + 4 * (q * w + 8 * (g % 4) + 4 * h + i);
    if (W >= 8 || h == 0) __builtin_nontemporal_store(f32x4{v[0], v[1], v[2], v[3]}, reinterpret_cast<f32x4*>(to));
  }
}

// Trilinear features of one record into the row order of the products: x[s] = feature tr_row(s, h) for
// the steps whose 8-row group holds features.  The loads are unconditional (empty corners read slot 0,
// which exists, and mask[q] zeroes their raw bits), so a group's eight loads are in flight together.
template <int F, bool HALF>
__device__ __forceinline__ void gather_rows(const void* __restrict__ feats, const Corners& cn, const uint32_t (&mask)[8],
                                            int h, float* x) {
  static_assert(F % 8 == 0 && F <= 32, "feature rows must fill whole 8-row groups of the first block");
#pragma unroll
  for (int g = 0; g < F / 8; ++g) {
    float v[8][4];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int64_t off = (int64_t)(cn.slot[q] >= 0 ? cn.slot[q] : 0) * F + 8 * g + 4 * h;
      if (HALF) {
        uint2 raw = *reinterpret_cast<const uint2*>(reinterpret_cast<const _Float16*>(feats) + off);
        raw.x &= mask[q];
        raw.y &= mask[q];
        const _Float16* hv = reinterpret_cast<const _Float16*>(&raw);
#pragma unroll
        for (int t = 0; t < 4; ++t) v[q][t] = (float)hv[t];
      } else {
        FeatLoad<false>::load(feats, off, mask[q], v[q]);
      }
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float qv[8] = {v[0][t], v[1][t], v[2][t], v[3][t], v[4][t], v[5][t], v[6][t], v[7][t]};
      x[4 * g + t] = tri_combine(qv, cn.wx, cn.wy, cn.wz);
    }
  }
}

}  // namespace snisr
