// Matrix-product building blocks of the FP32 training MLPs (the feature-scene training chain and the
// positional-encoding MLP): the packing of the weights, their staging through LDS and the product of one
// layer on v_mfma_f32_32x32x2_f32, and the splitting of the weight gradients' operands.
//
// The layer products take FP32 operands as they are and add them in one order (the bias, then the inputs in
// step order), so a value, an infinity and the sign of a hidden value near zero, which decides its ReLU, are
// what an FP32 chain gives.  Two-part FP16 operands with a power-of-two scale per layer were built and taken
// back, though they were faster (3.04M records at width 128: forward 1.15 ms against 2.45, backward 4.24
// against 5.90): they keep 22 bits, units far below their layer's largest weight lost bits and in the end
// vanished, an infinity became NaN and then 0 in the ReLU, and the other rounding of hidden values near zero
// moved the parameter gradients of the 530k-sample reflection step by 4e-5.
//
// Sums over records (the weight gradients) decide no sign: their operands are split into three BF16 parts,
// which keep the range and all 24 bits of FP32, and multiplied as six products (what is left out is below
// 2^-25).  An infinite operand, or one above the largest BF16 number (3.39e38), makes its row NaN.
#pragma once

#include "mfma_ops.hpp"
#include "snisr_device.hpp"

namespace snisr {

// One wavefront takes 32 records of one tile as the 32 columns, so every layer is W (out x in) times a
// 32-column block of activations.  Lane layouts of v_mfma_f32_32x32x2_f32 (h = lane / 32, c = lane % 32):
//   A:  lane holds A[row c][k = h]        B:  lane holds B[k = h][column c]
//   D:  lane holds rows 8(r/4) + 4h + (r%4), r = 0..15, of column c
// Register s of a lane's activations holds row tr_row(s, h): the order in which the D blocks of a layer
// come out.  Step s of a product pairs the rows tr_row(s, 0) and tr_row(s, 1), so its B operand is register s
// of the previous layer's output and activations never leave registers.  Layer 0's inputs (features, then
// the view encoding) follow the same row order.
__host__ __device__ constexpr int tr_row(int s, int h) { return 32 * (s / 16) + 8 * ((s % 16) / 4) + 4 * h + (s % 4); }
// registers of layer 0's inputs: whole 8-row groups
__host__ __device__ constexpr int tr_ns0(int in0) { return 16 * (in0 / 32) + 4 * ((in0 % 32 + 7) / 8); }

// Packed weights: a fragment is 32 output rows x 8 steps (16 inputs), as two pieces of 64 lanes x 4 steps; the
// fragments of a layer are ordered k-chunk by k-chunk, output block by output block, and padded to whole
// groups of kChunkFrags, the unit that is staged through LDS.  Order: the forward layers 0 .. L-1, the
// transposed layers L-1 .. 0, i.e. the order in which the kernels read them; then the biases (32 floats per
// output block, in the D layout).
constexpr int kPieceBytes = 1024, kFragBytes = 2 * kPieceBytes, kChunkFrags = 8, kChunkBytes = kChunkFrags * kFragBytes;
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
// float offset of layer l's biases in the packed block
__host__ __device__ constexpr int64_t tr_bias_off(int in0, int wd, int L, int l, int nout) {
  int64_t o = (int64_t)tr_bwd_chunk(in0, wd, L, -1, nout) * (kChunkBytes / 4);
  for (int m = 0; m < l; ++m) o += 32 * tr_nob(wd, L, m);
  return o;
}
// floats of a packed block
__host__ __device__ constexpr int64_t tr_stride(int in0, int wd, int L, int nout) {
  return (tr_bias_off(in0, wd, L, L, nout) + 63) / 64 * 64;
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
// One workgroup per layer and tile: the layer's forward and transposed fragments and its biases (mlp_params
// layout: per layer W[out][in], then b[out]; the last layer has nout <= 32 rows).
__device__ __forceinline__ void pack_train_layer(const float* __restrict__ P, float* __restrict__ block, int in0, int wd,
                                                 int L, int l, int nout) {
  for (int m = 0; m < l; ++m) P += (int64_t)((m == 0 ? in0 : wd) + 1) * wd;
  const int in = l == 0 ? in0 : wd, out = l == L - 1 ? nout : wd;
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
        const int o = bwd ? k : row, i = bwd ? row : k;
        v[e] = kc < nk && o < out && i < in ? P[(int64_t)o * in + i] : 0.0f;
      }
#pragma unroll
      for (int p = 0; p < 2; ++p)
        *reinterpret_cast<float4*>(to + (int64_t)f * kFragBytes + p * kPieceBytes + lane * 16) =
            make_float4(v[4 * p], v[4 * p + 1], v[4 * p + 2], v[4 * p + 3]);
    }
  }
}
}  // namespace

// The weight stream of a 256-thread workgroup: chunks of kChunkFrags fragments go from global memory
// through registers into one of two LDS buffers, the next chunk's loads in flight while the current one is
// used.  Without the staging every wavefront would read every fragment from L2 (2 KB per eight products).
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

// out(i, y) for register i of the NOB output blocks, y = bias + the layer's fragments times x, added in step
// order; x: registers s (row tr_row(s, h)) over NS steps; bias: NOB blocks of 32 floats, or NULL for zeros.  All
// output blocks advance together, so consecutive products are independent.
template <int NS, int NOB, class Out>
__device__ __forceinline__ void stream_layer(FragStream& fs, const float* x, int lane, const float* __restrict__ bias,
                                             Out out) {
  static_assert(kChunkFrags % NOB == 0 && NS % 4 == 0, "whole k-chunks per staged chunk, whole pieces");
  constexpr int KPC = kChunkFrags / NOB, NK = (NS + 7) / 8;
  f32x16 acc[NOB];
#pragma unroll
  for (int ob = 0; ob < NOB; ++ob) acc[ob] = bias ? bias_block(bias, ob, lane >> 5) : f32x16{};
#pragma unroll
  for (int k0 = 0; k0 < NK; k0 += KPC) {
    const uint8_t* A = fs.step() + lane * 16;
#pragma unroll
    for (int q = 0; q < 2 * KPC; ++q) {
      const int s = 8 * k0 + 4 * q;  // first of the four steps of piece q % 2 of k-chunk k0 + q / 2
      if (s >= NS) break;
      float4 a[NOB];
#pragma unroll
      for (int ob = 0; ob < NOB; ++ob)
        a[ob] = *reinterpret_cast<const float4*>(A + (q / 2 * NOB + ob) * kFragBytes + q % 2 * kPieceBytes);
#pragma unroll
      for (int ob = 0; ob < NOB; ++ob) acc[ob] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[ob].x, x[s], acc[ob], 0, 0, 0);
#pragma unroll
      for (int ob = 0; ob < NOB; ++ob) acc[ob] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[ob].y, x[s + 1], acc[ob], 0, 0, 0);
#pragma unroll
      for (int ob = 0; ob < NOB; ++ob) acc[ob] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[ob].z, x[s + 2], acc[ob], 0, 0, 0);
#pragma unroll
      for (int ob = 0; ob < NOB; ++ob) acc[ob] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[ob].w, x[s + 3], acc[ob], 0, 0, 0);
    }
  }
#pragma unroll
  for (int ob = 0; ob < NOB; ++ob)
#pragma unroll
    for (int r = 0; r < 16; ++r) out(16 * ob + r, acc[ob][r]);
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
// and features.  Cached | non-temporal, us: 530k samples of the reflection MLP, backward 522 | 495, dW 334 | 260; 3.04M
// records at width 128, backward 5587 | 5757, dW 2181 | 2126, the next forward 2415 | 2362 (equal in sum).
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
