// The reference's screen-space refinement U-Net (rendering/scripts/networks.py:5-73: ten 3x3
// convolutions with ReLU, 2x2 average pooling, bilinear x2 upsampling with align_corners and two
// channel concatenations; applied to the composited frame at rendering/src/__init__.py:336-339) on
// FP16 MFMA with FP32 accumulation.
//
// Activations are FP16 in planes of 16 channels: [channel / 16][pixel][channel % 16].  A convolution is
// an implicit GEMM: output channels are the rows (32-row blocks, the A operand of
// v_mfma_f32_32x32x16_f16), pixels the columns (a wavefront takes 64 consecutive pixels of a row as
// two 32-column blocks) and K runs over the 9 taps x 16-channel planes.  Lane (h, s) loads the B operand
// of one step as one 16-byte piece: channels 8h .. 8h + 7 of the plane at pixel s shifted by the tap, so
// the 64 lanes of a load cover 1 KB without a gap.  A concatenated input is two sources, chosen per plane,
// so the concatenation is never materialised.  The bias and ReLU are applied to the accumulators before
// the FP16 store.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mfma_ops.hpp"
#include "snisr_common.hpp"

namespace snisr {
namespace {

struct UnetLayer {
  int cin, cin_pad, cout, nob;
};
// conv1 .. conv10 of Unet (networks.py:8-15); cin_pad: channels rounded up to 16, nob: 32-row blocks
constexpr UnetLayer kUnet[10] = {{5, 16, 64, 2},    {64, 64, 32, 1},   {32, 32, 64, 2},  {64, 64, 64, 2},
                                 {64, 64, 128, 4},  {128, 128, 128, 4}, {192, 192, 64, 2}, {64, 64, 64, 2},
                                 {96, 96, 32, 1},   {32, 32, 3, 1}};

// packed layer: per output block ob, per step g = tap * (cin_pad / 16) + kc, a 1 KB A fragment
// (lane l = (h, s): W[32 ob + s][16 kc + 8 h + e][tap], e = 0..7, as FP16); then per output block
// the bias in accumulator order (32 floats)
__host__ __device__ constexpr int64_t unet_frag_bytes(int l) {
  return (int64_t)kUnet[l].nob * 9 * (kUnet[l].cin_pad / 16) * 1024;
}
__host__ __device__ constexpr int64_t unet_layer_bytes(int l) { return unet_frag_bytes(l) + kUnet[l].nob * 128; }
__host__ __device__ constexpr int64_t unet_layer_off(int l) {
  int64_t s = 0;
  for (int m = 0; m < l; ++m) s += unet_layer_bytes(m);
  return s;
}

__global__ void k_unet_pack_layer(const float* __restrict__ w, const float* __restrict__ b, uint8_t* __restrict__ dst,
                                  int l) {
  const UnetLayer L = kUnet[l];
  const int nkc = L.cin_pad / 16;
  const int64_t nfrag = (int64_t)L.nob * 9 * nkc;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nfrag * 64) {
    const int lane = (int)(i & 63), h = lane >> 5, s = lane & 31;
    const int64_t f = i >> 6;
    const int ob = (int)(f / (9 * nkc)), g = (int)(f % (9 * nkc)), tap = g / nkc, kc = g % nkc;
    const int co = 32 * ob + s;
    _Float16 v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int ci = 16 * kc + 8 * h + e;
      v[e] = (co < L.cout && ci < L.cin) ? (_Float16)w[((int64_t)co * L.cin + ci) * 9 + tap] : (_Float16)0.0f;
    }
    *reinterpret_cast<uint4*>(dst + f * 1024 + lane * 16) = *reinterpret_cast<const uint4*>(v);
  } else if (i < nfrag * 64 + L.nob * 32) {
    const int j = (int)(i - nfrag * 64), ob = j >> 5, h = (j >> 4) & 1, r = j & 15;
    const int co = 32 * ob + 8 * (r >> 2) + 4 * h + (r & 3);  // accumulator row of element r in lane half h
    reinterpret_cast<float*>(dst + unet_frag_bytes(l))[j] = co < L.cout ? b[co] : 0.0f;
  }
}

struct ConvArgs {
  const _Float16* src0;  // planes of input channels [0, C0)
  const _Float16* src1;  // planes of the remaining input channels (unused when src0 holds them all)
  int H, W;
  const uint8_t* layer;  // packed layer
  _Float16* dst;         // MODE 0: output planes
  float* out;            // MODE 1: [H, W, 3] float, min(ReLU(x), 1)
};

constexpr int kConvThreads = 512;

// One convolution; NKC input planes, the first C0 / 16 of them from src0; MODE 0: FP16 planes with ReLU, 1: the final
// three channels as min(ReLU(x), 1) in FP32.  A wavefront takes a strip of 64 pixels and sweeps down `rows` output
// rows: every B operand (one plane at one horizontal tap of one input row) is loaded once and multiplied by the three
// vertical taps, into the accumulators of the three output rows it belongs to; a row is finished, stored and its
// accumulators reused two input rows later.  One output block per workgroup (grid.y), its weights (9 * NKC KB) in LDS.
// Rows are read through buffer descriptors of one row of one plane, so pixels and rows outside the image read as
// zero without a branch; the loads run PD steps ahead, across the rows.
// What bounded the convolutions was the L1: a tap-by-tap kernel on channels-last pixels loaded each operand nine
// times, in 16-byte pieces 64 to 256 bytes apart.  All ten at 720 x 1280, summed: 880 us so; with one load for three
// taps, still channels-last, 700; with planes as well, whose loads are 1 KB of consecutive bytes, 363 (238 GFLOP with
// the padding of conv1 and conv10: 0.66 PFLOP/s).  Per layer, before and after: conv2 111 -> 40, conv7 228 -> 70, conv9
// 217 -> 69, conv10 44 -> 21, conv6 53 -> 33, conv1 54 -> 40 (its 118 MB of output at the copy rate: 23).  What is left
// is the two wavefronts per SIMD that the 96 accumulator registers and the ring allow.
template <int NKC, int C0, int MODE, int PD>
__global__ __launch_bounds__(kConvThreads, 2) void k_unet_conv(ConvArgs a, int rows) {
  using M = Mfma<SNISR_F16>;
  using vec = f16x8;
  constexpr int NS = 9 * NKC, NG = 3 * NKC;  // fragments; loads per input row (plane by plane, then horizontal tap)
  constexpr int R = PD + 1;
  static_assert(NG % R == 0, "the ring continues from row to row");
  extern __shared__ __align__(16) uint8_t lds[];
  const int ob = blockIdx.y;
  {
    const uint4* src = reinterpret_cast<const uint4*>(a.layer + (int64_t)ob * NS * 1024);
    uint4* dst = reinterpret_cast<uint4*>(lds);
    for (int k = threadIdx.x; k < NS * 64; k += blockDim.x) dst[k] = src[k];
    const float4* bs = reinterpret_cast<const float4*>(a.layer + (int64_t)gridDim.y * NS * 1024) + ob * 8;
    if (threadIdx.x < 8) reinterpret_cast<float4*>(lds + NS * 1024)[threadIdx.x] = bs[threadIdx.x];
  }
  __syncthreads();
  const float* bias = reinterpret_cast<const float*>(lds + NS * 1024);
  const int lane = threadIdx.x & 63, h = lane >> 5, s = lane & 31;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nwv = blockDim.x >> 6;
  const int H = a.H, W = a.W, strips = (W + 63) >> 6;
  const int tasks = strips * ((H + rows - 1) / rows);
  const uint8_t* Al = lds + lane * 16;
  const int64_t plane = (int64_t)H * W * 16;  // halves of one plane
  struct Row {
    const _Float16 *p0, *p1;  // the row in the first plane of each source
    int bytes;                // of the row in one plane; 0 outside the image
  };
  auto open_row = [&](int y) {
    const bool in = (unsigned)y < (unsigned)H;
    const int64_t r = (int64_t)(in ? y : 0) * W * 16;
    return Row{a.src0 + r, a.src1 + r, in ? W * 32 : 0};
  };
  for (int task = blockIdx.x * nwv + wv; task < tasks; task += gridDim.x * nwv) {
    const int x0 = task % strips * 64, y0 = task / strips * rows;
    const int y1 = y0 + rows < H ? y0 + rows : H;
    vec ring[R][2];
    auto load_b = [&](const Row& q, int g, int cb) -> vec {
      const int kc = g / 3, xx = x0 + 32 * cb + s + g % 3 - 1;  // left of the row: past every byte count
      const _Float16* p = 16 * kc < C0 ? q.p0 + kc * plane : q.p1 + (kc - C0 / 16) * plane;
      const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, q.bytes, 0x00027000);
      return __builtin_bit_cast(vec, __builtin_amdgcn_raw_buffer_load_b128(rsrc, xx * 32 + 16 * h, 0, 0));
    };
    Row cur = open_row(y0 - 1);
#pragma unroll
    for (int g = 0; g < PD; ++g) {
      ring[g][0] = load_b(cur, g, 0);
      ring[g][1] = load_b(cur, g, 1);
    }
    // input row y into the accumulators of output rows y - 1 (bottom taps), y and y + 1 (top taps); row y - 1
    // is complete after it (what rows outside y0 .. y1 - 1 collect is never stored)
    auto row = [&](int y, f32x16 (&up)[2], f32x16 (&mid)[2], f32x16 (&down)[2]) {
      const Row next = open_row(y + 1);
      vec w[2][3];
      const auto load_a = [&](int g, vec (&v)[3]) {
        const int kc = g / 3, dx = g % 3;
#pragma unroll
        for (int dy = 0; dy < 3; ++dy) v[dy] = load_frag<vec>(Al + ((3 * dy + dx) * NKC + kc) * 1024);
      };
      load_a(0, w[0]);
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        ring[(g + PD) % R][0] = g + PD < NG ? load_b(cur, g + PD, 0) : load_b(next, g + PD - NG, 0);
        ring[(g + PD) % R][1] = g + PD < NG ? load_b(cur, g + PD, 1) : load_b(next, g + PD - NG, 1);
        if (g + 1 < NG) load_a(g + 1, w[(g + 1) & 1]);
        const vec b0 = ring[g % R][0], b1 = ring[g % R][1];
        up[0] = M::mma(w[g & 1][2], b0, up[0]);
        mid[0] = M::mma(w[g & 1][1], b0, mid[0]);
        down[0] = M::mma(w[g & 1][0], b0, down[0]);
        up[1] = M::mma(w[g & 1][2], b1, up[1]);
        mid[1] = M::mma(w[g & 1][1], b1, mid[1]);
        down[1] = M::mma(w[g & 1][0], b1, down[1]);
        __builtin_amdgcn_sched_barrier(0);
      }
      cur = next;
      if (y - 1 >= y0) {
#pragma unroll
        for (int cb = 0; cb < 2; ++cb) {
          const int x = x0 + 32 * cb + s;
          const int64_t pix = (int64_t)(y - 1) * W + x;
          if (x < W) {
            if constexpr (MODE == 0) {
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                _Float16 v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                  const float t = up[cb][4 * j + r];
                  v[r] = (_Float16)(t > 0.0f ? t : 0.0f);
                }
                *reinterpret_cast<uint2*>(a.dst + (2 * ob + j / 2) * plane + pix * 16 + 8 * (j % 2) + 4 * h) =
                    *reinterpret_cast<const uint2*>(v);
              }
            } else if (h == 0) {
#pragma unroll
              for (int r = 0; r < 3; ++r) {
                const float t = up[cb][r];
                a.out[pix * 3 + r] = t > 0.0f ? (t < 1.0f ? t : 1.0f) : 0.0f;
              }
            }
          }
        }
      }
      up[0] = bias_block(bias, 0, h);
      up[1] = up[0];
    };
    f32x16 A[2], B[2], C[2];
    A[0] = bias_block(bias, 0, h);
    A[1] = B[0] = B[1] = C[0] = C[1] = A[0];
#pragma unroll 1
    for (int y = y0 - 1; y <= y1; y += 3) {
      row(y, A, B, C);
      if (y + 1 <= y1) row(y + 1, B, C, A);
      if (y + 2 <= y1) row(y + 2, C, A, B);
    }
  }
}

// One 16-byte piece (half a plane's channels of one output pixel) per thread; a row of pieces along grid.x, rows
// along grid.y, planes along grid.z, so no index is divided.

// 2x2 average pooling (nn.AvgPool2d(2, 2)), FP32 sum of the window in row order
__global__ void k_unet_pool(const _Float16* __restrict__ in, int Ho, int Wo, _Float16* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, xo = i >> 1, half = i & 1, W = 2 * Wo;
  if (xo >= Wo) return;
  const int64_t P = (int64_t)Ho * Wo;
  const _Float16* src = in + blockIdx.z * 4 * P * 16 + 8 * half;
  for (int yo = blockIdx.y; yo < Ho; yo += gridDim.y) {
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int dy = 0; dy < 2; ++dy)
#pragma unroll
      for (int dx = 0; dx < 2; ++dx) {
        const uint4 q = *reinterpret_cast<const uint4*>(src + ((int64_t)(2 * yo + dy) * W + 2 * xo + dx) * 16);
        const _Float16* hv = reinterpret_cast<const _Float16*>(&q);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = acc[e] + (float)hv[e];
      }
    _Float16 r[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = (_Float16)(acc[e] / 4.0f);
    *reinterpret_cast<uint4*>(out + (blockIdx.z * P + (int64_t)yo * Wo + xo) * 16 + 8 * half) = *reinterpret_cast<const uint4*>(r);
  }
}

// bilinear x2 upsampling with align_corners (nn.Upsample(scale_factor=2, mode="bilinear",
// align_corners=True)): source coordinate (in - 1) / (out - 1) * dst in FP32, the four neighbours
// weighted in the row-then-column order of the usual align-corners kernel
__global__ void k_unet_up(const _Float16* __restrict__ in, int Hi, int Wi, _Float16* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, xo = i >> 1, half = i & 1, Ho = 2 * Hi, Wo = 2 * Wi;
  if (xo >= Wo) return;
  const int64_t P = (int64_t)Ho * Wo;
  const _Float16* src = in + blockIdx.z * (P / 4) * 16 + 8 * half;
  const float sh = Ho > 1 ? (float)(Hi - 1) / (float)(Ho - 1) : 0.0f;
  const float sw = Wo > 1 ? (float)(Wi - 1) / (float)(Wo - 1) : 0.0f;
  const float wr = sw * (float)xo;
  const int w1 = (int)wr, wp = w1 < Wi - 1 ? 1 : 0;
  const float m1 = wr - (float)w1, m0 = 1.0f - m1;
  const auto px = [&](int yy, int xx) { return *reinterpret_cast<const f16x8*>(src + ((int64_t)yy * Wi + xx) * 16); };
  for (int yo = blockIdx.y; yo < Ho; yo += gridDim.y) {
    const float hr = sh * (float)yo;
    const int h1 = (int)hr, hp = h1 < Hi - 1 ? 1 : 0;
    const float l1 = hr - (float)h1, l0 = 1.0f - l1;
    const f16x8 a = px(h1, w1), b = px(h1, w1 + wp), c = px(h1 + hp, w1), d = px(h1 + hp, w1 + wp);
    f16x8 r;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      r[e] = (_Float16)(l0 * (m0 * (float)a[e] + m1 * (float)b[e]) + l1 * (m0 * (float)c[e] + m1 * (float)d[e]));
    *reinterpret_cast<f16x8*>(out + (blockIdx.z * P + (int64_t)yo * Wo + xo) * 16 + 8 * half) = r;
  }
}

// the 5-channel input (rgb, inverse depth, boundary flag; __init__.py:336-338) as one FP16 plane of 16 channels
__global__ void k_unet_input(const float* __restrict__ frame, const float* __restrict__ inv_near,
                             const uint8_t* __restrict__ boundary, int64_t n, _Float16* __restrict__ x16) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  _Float16 v[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) v[e] = (_Float16)0.0f;
  v[0] = (_Float16)frame[3 * i];
  v[1] = (_Float16)frame[3 * i + 1];
  v[2] = (_Float16)frame[3 * i + 2];
  v[3] = (_Float16)inv_near[i];
  v[4] = (_Float16)(boundary[i] ? 1.0f : 0.0f);
  uint4* d = reinterpret_cast<uint4*>(x16 + i * 16);
  d[0] = reinterpret_cast<const uint4*>(v)[0];
  d[1] = reinterpret_cast<const uint4*>(v)[1];
}

// workspace: the FP16 activations of every stage, 256-byte aligned
struct UnetWs {
  _Float16 *x16, *a1, *o2, *p1, *a3, *o5, *p2, *a5, *e7, *u7, *a7, *e4, *u9, *a9;
};

int64_t unet_ws(int64_t H, int64_t W, uint8_t* base, UnetWs* w) {
  const int64_t P = H * W, P2 = P / 4, P4 = P / 16;
  const int64_t halves[14] = {P * 16, P * 64, P * 32, P2 * 32, P2 * 64, P2 * 64, P4 * 64, P4 * 128,
                              P4 * 128, P2 * 128, P2 * 64, P2 * 64, P * 64, P * 32};
  _Float16** slots[14] = {&w->x16, &w->a1, &w->o2, &w->p1, &w->a3, &w->o5, &w->p2, &w->a5,
                          &w->e7,  &w->u7, &w->a7, &w->e4, &w->u9, &w->a9};
  int64_t off = 0;
  for (int k = 0; k < 14; ++k) {
    if (base) *slots[k] = reinterpret_cast<_Float16*>(base + off);
    off += (halves[k] * 2 + 255) & ~(int64_t)255;
  }
  return off;
}

template <int NKC, int C0, int MODE, int PD>
int conv_launch(int l, const _Float16* s0, const _Float16* s1, int H, int W, const uint8_t* packed, _Float16* dst,
                float* out, hipStream_t st) {
  static_assert(NKC * 16 <= 192 && C0 % 16 == 0 && C0 <= NKC * 16, "planes within the sources");
  const UnetLayer L = kUnet[l];
  const size_t lds = (size_t)9 * NKC * 1024 + 128;
  auto kern = k_unet_conv<NKC, C0, MODE, PD>;
  static bool lds_set = false;
  if (!lds_set) {
    SNISR_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    lds_set = true;
  }
  ConvArgs a;
  a.src0 = s0;
  a.src1 = s1;
  a.H = H;
  a.W = W;
  a.layer = packed + unet_layer_off(l);
  a.dst = dst;
  a.out = out;
  // Rows per task: a wavefront costs rows + 2 input rows and the launch that times the wavefronts per SIMD, of which two
  // fit and two are needed to cover each other's waits.  At 720 x 1280 this picks 8 rows for conv9 and conv2, 4 for
  // conv7 and 2 for conv6; measured with 3, 4 and 8 rows: conv9 94, 80, 69 us, conv7 99, 70, 91, conv6 37, 41, 57
  // (with 2: 33).
  const int64_t strips = (W + 63) / 64, simds = 4 * (int64_t)device_cus();
  int64_t rows = 2, best = 0;
  for (int64_t r = 2; r <= 16; ++r) {
    const int64_t waves = strips * ((H + r - 1) / r) * L.nob, deep = (waves + simds - 1) / simds;
    const int64_t cost = (deep > 2 ? deep : 2) * (r + 2);
    if (r == 2 || cost < best) {
      best = cost;
      rows = r;
    }
  }
  const int64_t tasks = strips * ((H + rows - 1) / rows), need = (tasks + kConvThreads / 64 - 1) / (kConvThreads / 64);
  const int per_cu = lds > 80 * 1024 ? 1 : 2;
  int64_t gx = ((int64_t)per_cu * device_cus() + L.nob - 1) / L.nob;
  gx = gx < need ? gx : need;
  hipLaunchKernelGGL(kern, dim3((unsigned)gx, (unsigned)L.nob), dim3(kConvThreads), lds, st, a, (int)rows);
  SNISR_LAUNCHED();
  return SNISR_OK;
}

// grid of a per-piece kernel over C channels of [H, W]
dim3 piece_grid(int H, int W, int C) {
  return dim3((unsigned)(((int64_t)2 * W + 255) / 256), (unsigned)(H < 65535 ? H : 65535), (unsigned)(C / 16));
}

int pool_launch(const _Float16* in, int H, int W, int C, _Float16* out, hipStream_t st) {
  hipLaunchKernelGGL(k_unet_pool, piece_grid(H / 2, W / 2, C), dim3(256), 0, st, in, H / 2, W / 2, out);
  SNISR_LAUNCHED();
  return SNISR_OK;
}

int up_launch(const _Float16* in, int Hi, int Wi, int C, _Float16* out, hipStream_t st) {
  hipLaunchKernelGGL(k_unet_up, piece_grid(2 * Hi, 2 * Wi, C), dim3(256), 0, st, in, Hi, Wi, out);
  SNISR_LAUNCHED();
  return SNISR_OK;
}

}  // namespace
}  // namespace snisr

using namespace snisr;

extern "C" {

int64_t snisr_unet_packed_size(void) { return unet_layer_off(10); }

int snisr_unet_pack(const float* const* weights, const float* const* biases, void* packed, void* stream) {
  SNISR_REQUIRE(weights && biases && packed, SNISR_ERR_ARG, "unet_pack: NULL pointer");
  SNISR_REQUIRE(aligned(packed, 256), SNISR_ERR_ALIGN, "unet_pack: packed must be 256-byte aligned");
  for (int l = 0; l < 10; ++l) {
    SNISR_REQUIRE(weights[l] && biases[l], SNISR_ERR_ARG, "unet_pack: layer %d has a NULL tensor", l);
    const int64_t n = unet_frag_bytes(l) / 16 + kUnet[l].nob * 32;
    hipLaunchKernelGGL(k_unet_pack_layer, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       weights[l], biases[l], (uint8_t*)packed + unet_layer_off(l), l);
    SNISR_LAUNCHED();
  }
  return SNISR_OK;
}

int64_t snisr_unet_workspace_size(int32_t H, int32_t W) {
  if (H <= 0 || W <= 0 || H % 4 || W % 4) {
    set_error("unet_workspace_size: H and W must be positive multiples of 4 (got %d x %d)", H, W);
    return -1;
  }
  return unet_ws(H, W, nullptr, nullptr);
}

int snisr_unet_refine(const void* packed, const float* frame, const float* inverse_near, const uint8_t* boundary,
                      int32_t H, int32_t W, void* workspace, int64_t workspace_bytes, float* out, void* stream) {
  SNISR_REQUIRE(H > 0 && W > 0 && H % 4 == 0 && W % 4 == 0, SNISR_ERR_SHAPE,
                "unet_refine: H and W must be positive multiples of 4 (got %d x %d)", H, W);
  SNISR_REQUIRE(packed && frame && inverse_near && boundary && workspace && out, SNISR_ERR_ARG,
                "unet_refine: NULL pointer");
  SNISR_REQUIRE(aligned(packed, 256) && aligned(workspace, 256), SNISR_ERR_ALIGN,
                "unet_refine: packed and workspace must be 256-byte aligned");
  SNISR_REQUIRE(workspace_bytes >= unet_ws(H, W, nullptr, nullptr), SNISR_ERR_CAPACITY,
                "unet_refine: workspace too small (snisr_unet_workspace_size)");
  UnetWs w;
  unet_ws(H, W, (uint8_t*)workspace, &w);
  const hipStream_t st = (hipStream_t)stream;
  const uint8_t* pk = (const uint8_t*)packed;
  const int64_t P = (int64_t)H * W;
  const int H2 = H / 2, W2 = W / 2, H4 = H / 4, W4 = W / 4;
  hipLaunchKernelGGL(k_unet_input, dim3((unsigned)((P + 255) / 256)), dim3(256), 0, st, frame, inverse_near, boundary,
                     P, w.x16);
  SNISR_LAUNCHED();
  int e;
  // o2 = relu(conv2(relu(conv1(x))))
  if ((e = conv_launch<1, 16, 0, 2>(0, w.x16, w.x16, H, W, pk, w.a1, nullptr, st))) return e;
  if ((e = conv_launch<4, 64, 0, 5>(1, w.a1, w.a1, H, W, pk, w.o2, nullptr, st))) return e;
  // o5 = relu(conv4(relu(conv3(down(o2)))))
  if ((e = pool_launch(w.o2, H, W, 32, w.p1, st))) return e;
  if ((e = conv_launch<2, 32, 0, 5>(2, w.p1, w.p1, H2, W2, pk, w.a3, nullptr, st))) return e;
  if ((e = conv_launch<4, 64, 0, 5>(3, w.a3, w.a3, H2, W2, pk, w.o5, nullptr, st))) return e;
  // e7 = relu(conv6(relu(conv5(down(o5)))))
  if ((e = pool_launch(w.o5, H2, W2, 64, w.p2, st))) return e;
  if ((e = conv_launch<4, 64, 0, 5>(4, w.p2, w.p2, H4, W4, pk, w.a5, nullptr, st))) return e;
  if ((e = conv_launch<8, 128, 0, 7>(5, w.a5, w.a5, H4, W4, pk, w.e7, nullptr, st))) return e;
  // e4 = relu(conv8(relu(conv7(cat(up(e7), o5)))))
  if ((e = up_launch(w.e7, H4, W4, 128, w.u7, st))) return e;
  if ((e = conv_launch<12, 128, 0, 5>(6, w.u7, w.o5, H2, W2, pk, w.a7, nullptr, st))) return e;
  if ((e = conv_launch<4, 64, 0, 5>(7, w.a7, w.a7, H2, W2, pk, w.e4, nullptr, st))) return e;
  // out = min(relu(conv10(relu(conv9(cat(up(e4), o2))))), 1)
  if ((e = up_launch(w.e4, H2, W2, 64, w.u9, st))) return e;
  if ((e = conv_launch<6, 64, 0, 5>(8, w.u9, w.o2, H, W, pk, w.a9, nullptr, st))) return e;
  if ((e = conv_launch<2, 32, 1, 5>(9, w.a9, w.a9, H, W, pk, nullptr, out, st))) return e;
  return SNISR_OK;
}

}  // extern "C"
