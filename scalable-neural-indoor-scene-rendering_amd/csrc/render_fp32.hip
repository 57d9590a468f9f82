// A1 camera rays, A2 tile DDA, and the plain FP32 renderer (march, FP32 MFMA MLP and compositing in one
// kernel, no workspace).
#include "mfma_ops.hpp"
#include "snisr_common.hpp"
#include "snisr_device.hpp"
#include "train_mma.hpp"

namespace snisr {

// ---------------------------------------------------------------------------- A1
// d = R [(px-cx)*invf, (py-cy)*invf, 1]   (rendering/src/compute_rays.cu:7-44)
__global__ __launch_bounds__(256) void k_compute_rays(const float* __restrict__ intr, const float* __restrict__ c2w,
                                                      int H, int W, float* __restrict__ rays_d) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)H * W) return;
  const int py = (int)(i / W), px = (int)(i - (int64_t)py * W);
  const float x = ((float)px - intr[0]) * intr[2];
  const float y = ((float)py - intr[1]) * intr[2];
#pragma unroll
  for (int r = 0; r < 3; ++r) rays_d[i * 3 + r] = c2w[3 * r] * x + c2w[3 * r + 1] * y + c2w[3 * r + 2];
}

// ---------------------------------------------------------------------------- A2
// One wave per 64 rays.  With STAGE, each lane writes its K entries into an LDS row (odd stride,
// so the 64 rows hit distinct banks) and the wave then stores the block's 64*K contiguous entries
// with coalesced writes; without it (K > kTraceStageMaxK) every lane writes its row directly.
constexpr int kTraceStageMaxK = 127;
template <bool STAGE>
__global__ __launch_bounds__(64) void k_trace_tiles(snisr_scene S, const float* __restrict__ origin,
                                                    const float* __restrict__ rays_d, int64_t n, int K,
                                                    int32_t* __restrict__ visited) {
  extern __shared__ int32_t trace_lds[];
  const int64_t base = (int64_t)blockIdx.x * 64;
  const int64_t i = base + threadIdx.x;
  const int KP = K | 1;
  if (i < n) {
    const V3 o = v3(origin[0], origin[1], origin[2]);
    const V3 d = v3(rays_d[3 * i], rays_d[3 * i + 1], rays_d[3 * i + 2]);
    TileWalker w;
    w.init(S, o, d, K);
    if (STAGE) {
      int32_t* row = trace_lds + threadIdx.x * KP;
      for (int j = 0; j < K; ++j) row[j] = w.next();
    } else {
      int32_t* out = visited + i * K;
      for (int j = 0; j < K; ++j) out[j] = w.next();
    }
  }
  if (!STAGE) return;
  __syncthreads();
  const int64_t rows = n - base < 64 ? n - base : 64;
  const int total = (int)rows * K;
  int32_t* out = visited + base * K;
  for (int q = threadIdx.x; q < total; q += 64) {
    const int r = q / K;
    out[q] = trace_lds[r * KP + (q - r * K)];
  }
}

// ---------------------------------------------------------------------------- MLP packing (f32t)
// mlp_params per tile: per layer W[out][in] then b[out]  ->  Wt[in][out4] then b[out4]
__global__ void k_pack_f32t(const float* __restrict__ src, int64_t src_stride, float* __restrict__ dst,
                            int64_t dst_stride, int in0, int width, int layers, int64_t total) {
  const int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= total) return;
  const int64_t tile = g / dst_stride;
  int64_t r = g - tile * dst_stride;
  const float* s = src + tile * src_stride;
  int in = in0;
  for (int l = 0; l < layers; ++l) {
    const int out = (l == layers - 1) ? 3 : width;
    const int o4 = (out + 3) & ~3;
    const int64_t wsz = (int64_t)in * o4;
    if (r < wsz) {
      const int i = (int)(r / o4), j = (int)(r - (int64_t)(r / o4) * o4);
      dst[g] = j < out ? s[(int64_t)j * in + i] : 0.0f;
      return;
    }
    r -= wsz;
    if (r < o4) {
      dst[g] = r < out ? s[(int64_t)out * in + r] : 0.0f;
      return;
    }
    r -= o4;
    s += (int64_t)out * in + out;
    in = out;
  }
}

// ---------------------------------------------------------------------------- FP32 render
// One wavefront takes 64 / kFp32Group rays, marched by groups of kFp32Group lanes (GroupMarch), and
// queues every sample's record in LDS; whenever 64 records are queued it evaluates their MLP together as
// the columns of v_mfma_f32_32x32x2_f32 products (activations in registers: the D layout of a layer is
// the B operand of the next, the weights read from the f32t packing, whose rows are the A operand's
// columns) and adds the weighted colours to their rays in sample order.
//
// What bounds it: the matrix products (12.5 kFLOP per sample at width 64).  The previous form ran one
// ray and one sample's MLP per lane on the vector units, re-reading every weight per sample and leaving
// most lanes idle once their rays had ended: 11.8 ms for the 320x180 single-tile view, 0.21 ms now; 85 ms
// for the 1280x720 frame of the 16-tile room, 10.1 ms now.  Eight lanes per ray: with 4 the small view takes
// 0.25 ms and the room 10.2, with 16 0.25 and 10.7 (more of the lanes past a brick's or ray's end).
constexpr int kFp32Group = 8, kFp32Rays = 64 / kFp32Group;

// acc += the product of one layer's f32t weights Wt[in][OUT4] with x over NS steps, all output blocks
// at once (consecutive products are independent); rows past the layer's ROWS inputs count as zero
template <int NS, int ROWS, int NOB, int CB, int OUT4>
__device__ __forceinline__ void f32t_product(const float* __restrict__ Wt, const float (*x)[64], int c, int h,
                                             f32x16 (&acc)[CB][NOB]) {
  constexpr int GS = 4;  // steps whose weights are loaded together, one such group ahead of the products
  float a[2][GS][NOB];
  // the lane's offset is hidden from the optimizer: the loads' addresses would otherwise be formed
  // once, outside the march loop, and held in registers
  int off = 4 * h * OUT4 + (c < OUT4 ? c : 0);
  asm volatile("" : "+v"(off));
  auto fetch = [&](int g, float (&v)[GS][NOB]) {
#pragma unroll
    for (int q = 0; q < GS; ++q)
#pragma unroll
      for (int ob = 0; ob < NOB; ++ob) {
        const float w = Wt[tr_row(g * GS + q, 0) * OUT4 + ob * 32 + off];
        const bool row_ok = tr_row(g * GS + q, 1) < ROWS || h == 0;  // lane half 1 holds the row 4 further on
        v[q][ob] = c < OUT4 && row_ok ? w : 0.0f;
      }
  };
  fetch(0, a[0]);
#pragma unroll
  for (int g = 0; g < NS / GS; ++g) {
    if (g + 1 < NS / GS) fetch(g + 1, a[(g + 1) & 1]);
#pragma unroll
    for (int q = 0; q < GS; ++q)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int ob = 0; ob < NOB; ++ob)
          acc[cb][ob] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g & 1][q][ob], x[cb][g * GS + q], acc[cb][ob], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// out = b (in the D layout) for NOB blocks of CB column blocks
template <int NOB, int CB>
__device__ __forceinline__ void f32t_bias(const float* __restrict__ b, int h, f32x16 (&acc)[CB][NOB]) {
#pragma unroll
  for (int ob = 0; ob < NOB; ++ob)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 v = *reinterpret_cast<const float4*>(b + 32 * ob + 8 * q + 4 * h);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        acc[cb][ob][4 * q] = v.x;
        acc[cb][ob][4 * q + 1] = v.y;
        acc[cb][ob][4 * q + 2] = v.z;
        acc[cb][ob][4 * q + 3] = v.w;
      }
    }
}

// The MLP of CB blocks of 32 columns in one tile: x[cb] the layer-0 inputs in step order (overwritten),
// z[cb][0..2] the output pre-activations (lanes of half 0)
template <int IN, int WD, int L, int CB>
__device__ __forceinline__ void f32t_mlp(const float* __restrict__ P, float (*x)[64], int c, int h, float (*z)[3]) {
  constexpr int NOB = WD / 32;
  auto relu_into = [&](f32x16(&acc)[CB][NOB]) {
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int r = 0; r < 16 * NOB; ++r) x[cb][r] = acc[cb][r / 16][r % 16] > 0.0f ? acc[cb][r / 16][r % 16] : 0.0f;
  };
  {
    f32x16 acc[CB][NOB];
    f32t_bias<NOB, CB>(P + IN * WD, h, acc);
    f32t_product<tr_ns0(IN), IN, NOB, CB, WD>(P, x, c, h, acc);
    relu_into(acc);
  }
  P += IN * WD + WD;
#pragma unroll 1
  for (int l = 1; l < L - 1; ++l) {
    f32x16 acc[CB][NOB];
    f32t_bias<NOB, CB>(P + WD * WD, h, acc);
    f32t_product<WD / 2, WD, NOB, CB, WD>(P, x, c, h, acc);
    relu_into(acc);
    P += WD * WD + WD;
  }
  f32x16 acc[CB][1];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) acc[cb][0] = f32x16{};
  f32t_product<WD / 2, WD, 1, CB, 4>(P, x, c, h, acc);
#pragma unroll
  for (int cb = 0; cb < CB; ++cb)
#pragma unroll
    for (int i = 0; i < 3; ++i) z[cb][i] = acc[cb][0][i] + P[WD * 4 + i];
}

// two waves per SIMD at least: one wave's march waits while the other's products run
template <int F, int WD, int L, bool HALF>
__global__ __launch_bounds__(64, 2) void k_render_fp32(snisr_scene S, snisr_march_params P, snisr_rays R,
                                                    snisr_render_out O, int packet_w) {
  constexpr int G = kFp32Group, RPW = 64 / G, IN = F + 15, NS0 = tr_ns0(IN), QCAP = 128;
  constexpr int CB = WD <= 64 ? 2 : 1;  // column blocks per pass of the MLP (registers at width 128)
  static_assert(WD % 32 == 0 && WD <= 128 && F % 8 == 0 && F <= 32 && NS0 <= 64, "MLP shape");
  __shared__ float4 q_rec[QCAP];        // voxel coordinate, compositing weight
  __shared__ int q_tile[QCAP], q_ray[QCAP];
  __shared__ float enc_lds[RPW][17];
  __shared__ float res[64][3];          // weighted colours of the batch
  const int lane = threadIdx.x, c = lane & 31, h = lane >> 5;
  const int rl = lane / G;              // this lane's ray within the wavefront
  const int64_t tid = (int64_t)blockIdx.x * RPW + rl;
  constexpr int64_t wstride = f32t_stride(IN, WD, L);
  const bool has = tid < R.n;
  const int64_t i = has ? ray_of_thread(tid, R.n, packet_w) : 0;
  GroupMarch<G> m;
  m.phase = GroupMarch<G>::kDone;
  int32_t* bricks = has && O.bricks ? O.bricks + i * O.brick_cap : nullptr;
  if (has) {
    const float* og = R.origins + i * R.origin_stride;
    const V3 d = normalize_dir(v3(R.dirs[3 * i], R.dirs[3 * i + 1], R.dirs[3 * i + 2]));
    m.init(S, P, v3(og[0], og[1], og[2]), d, R.t_hit ? R.t_hit[i] : __builtin_inff(),
           R.visited ? R.visited + i * P.max_tiles : nullptr);
    if (lane % G == 0) {
      float enc[15];
      view_encoding(d, enc);
#pragma unroll
      for (int k = 0; k < 15; ++k) enc_lds[rl][k] = enc[k];
    }
  }
  // lane 3 r + ch < 3 RPW sums channel ch of ray r
  float col = 0.0f;
  int qn = 0;  // queued records (wave-uniform)
  auto sync = [&] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  // evaluates the first nq <= 64 queued records and adds their colours
  auto shade = [&](int nq) {
    sync();
    uint64_t todo = nq >= 64 ? ~0ull : (1ull << nq) - 1;
    const int own_tile = lane < nq ? q_tile[lane] : -1;
    // one pass per distinct tile among the records (nearly always one)
    while (todo) {
      const int t = __builtin_amdgcn_readlane(own_tile, __builtin_ctzll(todo));
      const uint64_t in_t = __builtin_amdgcn_ballot_w64(own_tile == t);
      todo &= ~in_t;
#pragma unroll 1
      for (int c0 = 0; c0 < 2; c0 += CB) {
        if (!((in_t >> (32 * c0)) & (CB == 2 ? ~0ull : 0xffffffffull))) continue;
        float x[CB][64];
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
          const int r = 32 * (c0 + cb) + c;
          const bool ok = in_t >> r & 1;
          const float4 rec = ok ? q_rec[r] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
          Corners cn;
          find_corners(S.brick_map + S.tile_brick_base[t], S.tile_res[t], v3(rec.x, rec.y, rec.z), cn);
          uint32_t mask[8];
#pragma unroll
          for (int k = 0; k < 8; ++k) mask[k] = corner_mask(ok && cn.slot[k] >= 0);
          gather_rows<F, HALF>(S.feats, cn, mask, h, x[cb]);
          __builtin_amdgcn_sched_barrier(0);  // one block's corner rows in registers at a time
          const float* e = enc_lds[ok ? q_ray[r] : 0];
#pragma unroll
          for (int s = 0; s < NS0; ++s) {
            const int r0 = tr_row(s, 0) - F, r1 = tr_row(s, 1) - F;  // encoding entry of each half
            if (r0 >= 0) x[cb][s] = h ? (r1 < 15 ? e[r1 < 15 ? r1 : 0] : 0.0f) : (r0 < 15 ? e[r0 < 15 ? r0 : 0] : 0.0f);
          }
        }
        float z[CB][3];
        f32t_mlp<IN, WD, L, CB>(S.mlp_f32t + (int64_t)t * wstride, x, c, h, z);
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
          const int r = 32 * (c0 + cb) + c;
          if (h == 0 && (in_t >> r & 1)) {
            const float w = q_rec[r].w;
#pragma unroll
            for (int k = 0; k < 3; ++k) res[r][k] = w * sigmoid_cw(z[cb][k]);
          }
        }
      }
    }
    sync();
    if (lane < 3 * RPW) {
      const int ray = lane / 3, ch = lane - 3 * ray;
      for (int r = 0; r < nq; ++r)
        if (q_ray[r] == ray) col = col + res[r][ch];
    }
    sync();
  };
  while (true) {
    const bool live = m.phase != GroupMarch<G>::kDone;
    const bool marching = __builtin_amdgcn_ballot_w64(live) != 0;
    if (!marching && qn == 0) break;
    float4 rec;
    int tile = 0;
    bool took = false;
    if (live) {
      const bool turn = tile_quorum(m.phase == GroupMarch<G>::kTile);
      took = m.step(S, P, turn, bricks, O.brick_cap,
                    [&](int t, const V3& f, const Corners&, float w, float, float, float, int) {
                      rec = make_float4(f.x, f.y, f.z, w);
                      tile = t;
                    });
    }
    // a ray's samples of one step sit on consecutive lanes, so the queue keeps every ray's order
    const uint64_t tm = __builtin_amdgcn_ballot_w64(took);
    if (took) {
      const int at = qn + __builtin_popcountll(tm & ((1ull << lane) - 1));
      q_rec[at] = rec;
      q_tile[at] = tile;
      q_ray[at] = rl;
    }
    qn += __builtin_popcountll(tm);
    if (qn >= 64 || !marching) {  // a full batch, or what is left at the end
      const int nq = qn < 64 ? qn : 64;
      shade(nq);
      qn -= nq;
      if (lane < qn) {  // fewer than 64 remain: they move to the front
        q_rec[lane] = q_rec[64 + lane];
        q_tile[lane] = q_tile[64 + lane];
        q_ray[lane] = q_ray[64 + lane];
      }
    }
  }
  if (has && lane % G == 0) {
    if (bricks)
      for (int k = m.nbr; k < O.brick_cap; ++k) bricks[k] = -1;
    if (O.T) O.T[i] = m.T;
    if (O.n_samples) O.n_samples[i] = m.nsamp;
    if (O.depth) O.depth[i] = m.depth;
  }
  if (lane < 3 * RPW) {
    const int64_t t = (int64_t)blockIdx.x * RPW + lane / 3;
    if (t < R.n) O.rgb[3 * ray_of_thread(t, R.n, packet_w) + lane % 3] = col;
  }
}

// sigma-only march (no MLP): counts, T, depth, bricks; used when rgb is not requested.
__global__ __launch_bounds__(64) void k_march_sigma(snisr_scene S, snisr_march_params P, snisr_rays R,
                                                    snisr_render_out O, int packet_w) {
  const int64_t tid = (int64_t)blockIdx.x * 64 + threadIdx.x;
  if (tid >= R.n) return;
  const int64_t i = ray_of_thread(tid, R.n, packet_w);
  const float* og = R.origins + i * R.origin_stride;
  const V3 origin = v3(og[0], og[1], og[2]);
  const V3 d = normalize_dir(v3(R.dirs[3 * i], R.dirs[3 * i + 1], R.dirs[3 * i + 2]));
  const float t_hit = R.t_hit ? R.t_hit[i] : __builtin_inff();
  int32_t* bricks = O.bricks ? O.bricks + i * O.brick_cap : nullptr;
  MarchResult res;
  march_ray(S, P, origin, d, t_hit, R.visited ? R.visited + i * P.max_tiles : nullptr, bricks, O.brick_cap,
            [&](int, const V3&, const Corners&, float, float, float, float) {}, res);
  if (bricks)
    for (int k = res.n_bricks; k < O.brick_cap; ++k) bricks[k] = -1;
  if (O.T) O.T[i] = res.T;
  if (O.n_samples) O.n_samples[i] = res.n_samples;
  if (O.depth) O.depth[i] = res.depth;
}

int packet_width(const snisr_rays& R) {
  if (R.image_width <= 0 || R.image_width % 8 != 0) return 0;
  if (R.n % R.image_width != 0) return 0;
  const int64_t rows = R.n / R.image_width;
  return rows % 8 == 0 ? R.image_width : 0;
}

}  // namespace snisr

using namespace snisr;

extern "C" {

int snisr_compute_rays(const float* intrinsic, const float* c2w, int32_t H, int32_t W, float* rays_d,
                       void* stream) {
  SNISR_REQUIRE(intrinsic && c2w && rays_d, SNISR_ERR_ARG, "compute_rays: NULL pointer");
  SNISR_REQUIRE(H >= 0 && W >= 0, SNISR_ERR_ARG, "compute_rays: negative size");
  const int64_t n = (int64_t)H * W;
  if (n == 0) return SNISR_OK;
  hipLaunchKernelGGL(k_compute_rays, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     intrinsic, c2w, H, W, rays_d);
  SNISR_LAUNCHED();
  return SNISR_OK;
}

int snisr_trace_tiles(const snisr_scene* scene, const float* origin, const float* rays_d, int64_t n, int32_t K,
                      int32_t* visited, void* stream) {
  // only the tile grid is read: tile_shape, scene_min, tile_size, tile_index_map
  SNISR_REQUIRE(scene, SNISR_ERR_ARG, "scene descriptor is NULL");
  SNISR_REQUIRE(scene->tile_shape[0] > 0 && scene->tile_shape[1] > 0 && scene->tile_shape[2] > 0, SNISR_ERR_ARG,
                "tile_shape must be positive");
  SNISR_REQUIRE(scene->tile_size > 0.0f, SNISR_ERR_ARG, "tile_size must be positive");
  SNISR_REQUIRE(scene->tile_index_map, SNISR_ERR_ARG, "tile_index_map is NULL");
  SNISR_REQUIRE(origin && (n == 0 || (rays_d && visited)), SNISR_ERR_ARG, "trace_tiles: NULL pointer");
  SNISR_REQUIRE(n >= 0 && K >= 0, SNISR_ERR_ARG, "trace_tiles: negative size");
  if (n == 0 || K == 0) return SNISR_OK;
  const dim3 grid((unsigned)((n + 63) / 64));
  if (K <= kTraceStageMaxK)
    hipLaunchKernelGGL(k_trace_tiles<true>, grid, dim3(64), (size_t)64 * (K | 1) * sizeof(int32_t),
                       (hipStream_t)stream, *scene, origin, rays_d, n, K, visited);
  else
    hipLaunchKernelGGL(k_trace_tiles<false>, grid, dim3(64), 0, (hipStream_t)stream, *scene, origin, rays_d, n, K,
                       visited);
  SNISR_LAUNCHED();
  return SNISR_OK;
}

int snisr_render_fp32(const snisr_scene* scene, const snisr_march_params* params, const snisr_rays* rays,
                      const snisr_render_out* out, void* stream) {
  SNISR_REQUIRE(out, SNISR_ERR_ARG, "render_fp32: out is NULL");
  const bool want_rgb = out->rgb != nullptr;
  if (int e = check_scene(scene, want_rgb)) return e;
  if (int e = check_params(params)) return e;
  if (int e = check_rays(rays, params)) return e;
  SNISR_REQUIRE(!out->bricks || out->brick_cap > 0, SNISR_ERR_ARG, "render_fp32: bricks needs brick_cap > 0");
  if (rays->n == 0) return SNISR_OK;
  const int pw = packet_width(*rays);
  const dim3 grid((unsigned)((rays->n + 63) / 64));
  hipStream_t st = (hipStream_t)stream;
  if (!want_rgb) {
    SNISR_HIP(stage_event(out, 0, st));
    hipLaunchKernelGGL(k_march_sigma, grid, dim3(64), 0, st, *scene, *params, *rays, *out, pw);
    SNISR_LAUNCHED();
    SNISR_HIP(stage_event(out, 1, st));
    return SNISR_OK;
  }
  SNISR_REQUIRE(scene->mlp_f32t, SNISR_ERR_ARG, "render_fp32: scene.mlp_f32t is NULL (snisr_pack_mlp(SNISR_F32))");
  SNISR_REQUIRE(aligned(scene->mlp_f32t, 16), SNISR_ERR_ALIGN, "render_fp32: mlp_f32t must be 16-byte aligned");
  const int F = scene->feat_dim, WD = scene->mlp_width, L = scene->mlp_layers;
  const bool half = scene->feat_dtype == SNISR_F16;
#define SNISR_FP32_CASE(F_, W_, L_, H_)                                                                   \
  if (F == F_ && WD == W_ && L == L_ && half == H_) {                                                     \
    SNISR_HIP(stage_event(out, 0, st));                                                                   \
    hipLaunchKernelGGL((k_render_fp32<F_, W_, L_, H_>), dim3((unsigned)((rays->n + kFp32Rays - 1) / kFp32Rays)), \
                       dim3(64), 0, st, *scene, *params, *rays, *out, pw);                                \
    SNISR_LAUNCHED();                                                                                     \
    SNISR_HIP(stage_event(out, 1, st));                                                                   \
    return SNISR_OK;                                                                                      \
  }
  SNISR_FP32_CASE(16, 64, 3, false)
  SNISR_FP32_CASE(16, 64, 3, true)
  SNISR_FP32_CASE(32, 128, 4, true)
  SNISR_FP32_CASE(32, 128, 4, false)
  SNISR_FP32_CASE(16, 32, 3, false)
#undef SNISR_FP32_CASE
  set_error("render_fp32: unsupported shape F=%d width=%d layers=%d feat_dtype=%d", F, WD, L, scene->feat_dtype);
  return SNISR_ERR_SHAPE;
}

int64_t snisr_pack_mlp_size(const snisr_scene* scene, int32_t dtype) {
  if (!scene) return -1;
  if (dtype == SNISR_F32)
    return (int64_t)scene->n_tiles * mlp_f32t_stride(scene->mlp_in, scene->mlp_width, scene->mlp_layers) * 4;
  return mfma_pack_bytes(scene, dtype);
}

int snisr_pack_mlp(const snisr_scene* scene, int32_t dtype, void* packed, void* stream) {
  SNISR_REQUIRE(scene && packed && scene->mlp_params, SNISR_ERR_ARG, "pack_mlp: NULL pointer");
  SNISR_REQUIRE(scene->n_tiles > 0 && scene->mlp_layers >= 2, SNISR_ERR_ARG, "pack_mlp: bad MLP shape");
  if (dtype == SNISR_F32) {
    const int64_t ds = mlp_f32t_stride(scene->mlp_in, scene->mlp_width, scene->mlp_layers);
    const int64_t total = ds * scene->n_tiles;
    hipLaunchKernelGGL(k_pack_f32t, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       scene->mlp_params, scene->mlp_stride, (float*)packed, ds, scene->mlp_in, scene->mlp_width,
                       scene->mlp_layers, total);
    SNISR_LAUNCHED();
    return SNISR_OK;
  }
  return mfma_pack(scene, dtype, packed, stream);
}

}  // extern "C"
