#!/usr/bin/env python3
"""Benchmark: full-frame render of the 16-tile synthetic room (1280x720) on one MI355X.

One step = one frame through the hot path with every input resident in HBM:
camera rays -> BVH nearest hit on the 200k-triangle proxy mesh (bounds the march) -> tile DDA,
brick DDA march and sigma compositing -> per-tile width-128x4 MLP on FP16 MFMA with FP32
accumulation -> ordered per-ray reduction.  The timed steps replay the step captured once in a HIP
graph; per-stage kernel times come from eager steps with HIP events between the stages.  Further
legs (plain FP32 path, C3 training, the reference-format FRender pipeline, C4 batched uneven tiles,
C5 large scene, CPU oracle baseline) add fields to the same JSON line.
"""
from __future__ import annotations

import argparse
import json
import os
import sys
import time

REPO = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(REPO, "scalable-neural-indoor-scene-rendering_amd"))

METRIC = "Mrays/s render (1280x720) & train fwd+bwd at PSNR>=50dB vs FP64, 1 MI355X"
MFMA_PEAK_F16_TFLOPS = 2500.0   # MI355X dense FP16 MFMA
MFMA_PEAK_F32_TFLOPS = 157.3    # MI355X dense FP32 MFMA
HBM_PEAK_GBS = 8000.0
# HBM bytes per k_mlp_mfma launch on this workload: rocprofv3 FETCH_SIZE x 2.0 + WRITE_SIZE x 1.0
# (factors from a 256 MiB device copy), see profiles/c2_render_kernels.md
MLP_HBM_BYTES_PER_LAUNCH = 217.9e6 + 129.5e6

_T0 = time.perf_counter()


def progress(msg: str) -> None:
    """One line on stderr per finished leg (stdout carries only the result line)."""
    print(f"[bench {time.perf_counter() - _T0:7.1f} s] {msg}", file=sys.stderr, flush=True)

def mlp_flops_per_sample(mlp_in, width, layers):
    from snisr.scene import mlp_layer_dims
    return 2 * sum(i * o for i, o in mlp_layer_dims(mlp_in, width, layers))


def cpu_baseline(sc, cam, dirs_np, t_hit_np, frac, seed=0):
    """The oracle (FP32, OpenMP over all host cores) on a seeded subset of the frame's rays,
    given the GPU's mesh t_hit (the CPU mesh query is not part of the timed sample)."""
    import numpy as np
    sys.path.insert(0, os.path.join(REPO, "oracle"))
    import oracle as O
    O.build()
    osc = O.OracleScene(sc)
    n = dirs_np.shape[0]
    idx = np.sort(np.random.default_rng(seed).choice(n, max(1, int(n * frac)), replace=False))
    O.render(osc, cam.origin, dirs_np, t_hit=t_hit_np, ray_index=idx[:256])  # warm-up
    t0 = time.perf_counter()
    O.render(osc, cam.origin, dirs_np, t_hit=t_hit_np, ray_index=idx)
    dt = time.perf_counter() - t0
    cores = O.num_threads()
    return dict(value=round(len(idx) / dt / 1e6, 4), unit="Mrays/s", cores=cores, kind="port",
                sample=f"{len(idx)} seeded rays ({frac:.0%} of the 1280x720 frame), FP32 oracle march+MLP+"
                       f"compositing with the GPU mesh t_hit, {dt:.2f} s wall on {cores} threads "
                       f"({dt * cores:.0f} core-seconds)")


def psnr_vs_fp64(sc, cam, dirs_np, t_hit_np, rgb_gpu, n_rays=2000, seed=1):
    import numpy as np
    sys.path.insert(0, os.path.join(REPO, "oracle"))
    import oracle as O
    idx = np.sort(np.random.default_rng(seed).choice(dirs_np.shape[0], n_rays, replace=False))
    ref = O.render(O.OracleScene(sc), cam.origin, dirs_np, t_hit=t_hit_np, ray_index=idx, precision="f64")
    mse = float(np.mean((rgb_gpu[idx].astype(np.float64) - ref["rgb"].astype(np.float64)) ** 2))
    return 10 * np.log10(1.0 / max(mse, 1e-30))


def train_bench(args, dev):
    """C3: one training step = forward + backward (hand-written adjoint) + Adam on the 16-tile
    scene with FP32 features/MLP, 8192 rays per tile (131,072 rays), MSE against the render of a
    perturbed copy."""
    import numpy as np
    import torch
    from snisr import device as D
    from snisr import scene as S
    from snisr import train as TR

    sc, _, _ = S.config_c2(n_triangles=0, H=8, W=8, feat_half=False)
    tgt_sc = S.perturbed_copy(sc, 3)
    origins_np, dirs_np = S.config_c3_rays(sc, 3, 8192)
    o = torch.from_numpy(origins_np).to(dev)
    d = torch.from_numpy(dirs_np).to(dev)
    ds_t = D.DeviceScene(tgt_sc)
    with torch.no_grad():
        target, _ = TR.train_forward(ds_t, o, d)
        target = target["rgb"].clone()
    del ds_t
    ds = D.DeviceScene(sc)
    sigma = ds.sigma.clone().requires_grad_(True)
    feats = ds.feats.clone().requires_grad_(True)
    mlp = ds.mlp_params.clone().requires_grad_(True)
    opt = TR.Adam([sigma, feats, mlp], lr=1e-4)   # one-pass HIP Adam (torch.optim.Adam semantics)
    ws = TR.TrainWorkspace()
    losses = []

    def step():
        opt.zero_grad(set_to_none=True)
        rgb = TR.render(sigma, feats, mlp, o, d, ds, workspace=ws)
        loss = torch.mean((rgb - target) ** 2)
        loss.backward()
        opt.step()
        return loss

    for _ in range(2):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.train_steps):
        losses.append(step().detach())
    torch.cuda.synchronize()
    ms = (time.perf_counter() - t0) * 1e3 / args.train_steps
    n = o.shape[0]
    samples = int(ws.samples_last())
    # forward + backward of the MLP = 3 x the forward FLOPs per sample (the layer products on FP32 MFMA; the weight
    # gradients run as six BF16 products, so the FP32 MFMA peak is a yardstick for them, not a bound)
    tflops = 3 * samples * mlp_flops_per_sample(sc.mlp_in, sc.mlp_width, sc.mlp_layers) / (ms * 1e-3) / 1e12
    return {"train_mrays_s": round(n / (ms * 1e-3) / 1e6, 3), "train_ms_per_step": round(ms, 3),
            "train_samples_per_step": samples,
            "train_roofline": dict(bound="mfma", dtype="f32", achieved=round(tflops, 1),
                                   peak=MFMA_PEAK_F32_TFLOPS, unit="TFLOP/s",
                                   frac=round(tflops / MFMA_PEAK_F32_TFLOPS, 4),
                                   note="3 x 78,336 FLOP per sample over the whole step (fwd, adjoint, Adam)"),
            "train_rays_per_step": int(n), "train_loss_first_last": [float(losses[0]), float(losses[-1])],
            "train_config": "C3: C2 scene with FP32 features/MLP, 16 tiles x 8192 rays, MSE vs a perturbed "
                            "copy, fwd + hand-written adjoint + Adam (lr 1e-4)"}


def ref_train_bench(args, dev):
    """The reference's tile training step, Tile.train_batch (training/scripts/tile/tile.py:631-785),
    at its configuration (training/config/cfg.yaml: NUM_VOXEL 64, VOXEL_SIZE 0.02, one 91 x 91 patch,
    NSAMPLES 64, BGSAMPLE 32 over BGSAMPLE_RANGE 0.5, RSAMPLES 64, surface MLP 8 x 64 ReLU, reflection
    MLP 6 x 64 LeakyReLU, SH degree 2), on synthetic data: 15% of the dilated 66^3 nodes occupied,
    rays from around the tile through it with a background depth behind it.  One step = the
    samplers, the forward of train_FLAG 0 (diffuse), 1 (specular) or 2 (both), a masked MSE, the
    adjoints and Adam on both MLPs."""
    import numpy as np
    import torch
    from snisr import tile_train as TT
    from snisr import train as TRN
    from snisr import train_ref as TR

    rng = np.random.default_rng(5)
    NV, vs, P, S, NB, RS = 64, 0.02, 91, 64, 32, 64
    D, tile_size, n = NV + 2, NV * vs, P * P
    tc = np.zeros(3)
    flags = torch.tensor(np.where(rng.uniform(0, 1, (D, D, D)) < 0.15, 1, -1).astype(np.int16), device=dev)
    tile = TT.TileState(nodes_flag=flags, num_voxel=NV, voxel_size=vs, tile_center=tuple(tc), group_center=(0.0, 0.0, 0.0),
                        group_size=4.0, far=8.0)
    o = tc + rng.normal(size=(n, 3)) / np.sqrt(3) * 1.6 * tile_size
    tgt = tc + rng.uniform(-0.45, 0.45, (n, 3)) * tile_size
    d = tgt - o
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    bgd = np.linalg.norm(tgt - o, axis=1, keepdims=True) + tile_size * rng.uniform(0.6, 1.5, (n, 1))
    batch = np.concatenate([o, d, bgd, rng.uniform(0, 1, (n, 6)), np.ones((n, 1))], 1).reshape(1, P, P, 14)
    batch = torch.tensor(batch.astype(np.float32), device=dev)
    surf, refl = TR.PEMLP(8, 4, 0.0, device=dev), TR.PEMLP(6, 28, 0.01, device=dev)
    torch.manual_seed(0)
    with torch.no_grad():
        for m in (surf, refl):
            m.params.normal_(0.0, 0.1)
    opt = TRN.Adam([surf.params, refl.params], lr=1e-4)

    def step(flag):
        opt.zero_grad(set_to_none=True)
        out = TT.train_batch_forward(tile, surf, refl, batch, flag, S, NB, RS, 0.5, P)
        m = out["mask"]
        loss = (((out["pred"] - out["gtcolor"]) ** 2) * m).sum() / m.sum()
        loss.backward()
        opt.step()

    res = {}
    for flag in (0, 1, 2):
        for _ in range(2):
            step(flag)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(args.ref_train_steps):
            step(flag)
        torch.cuda.synchronize()
        ms = (time.perf_counter() - t0) * 1e3 / args.ref_train_steps
        res[f"ref_train_flag{flag}_ms_per_step"] = round(ms, 3)
        res[f"ref_train_flag{flag}_mrays_s"] = round(n / (ms * 1e-3) / 1e6, 3)
    # the four training samplers alone (utils.py:786-820) on the same batch; the reflection sampler
    # reads the grid the last diffuse step baked
    rays_o = batch[..., :3].reshape(-1, 3).contiguous()
    rays_d = batch[..., 3:6].reshape(-1, 3).contiguous()
    bgdepth = batch[..., 6:7].reshape(-1, 1).contiguous()
    inner = tile.nodes_flag[1:-1, 1:-1, 1:-1]
    samplers = {
        "sparse": lambda: TT.sparse_sampling(rays_o, rays_d, inner, NV, tile.tile_center, tile.tile_size, S),
        "background": lambda: TT.sampling_background(rays_o, rays_d, bgdepth, tile.tile_center, tile.tile_size, NB,
                                                     0.5),
        "uniform": lambda: TT.uniform_sampling(rays_o, rays_d, tile.tile_center, tile.tile_size, S),
        "reflection": lambda: TT.reflection_sampling(rays_o, rays_d, inner, tile.voxels, NV, tile.tile_center,
                                                     tile.tile_size, RS, tile.far, 1.0),
    }
    for name, fn in samplers.items():
        fn()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(20):
            fn()
        torch.cuda.synchronize()
        res[f"sampler_{name}_ms"] = round((time.perf_counter() - t0) * 1e3 / 20, 4)
    res["ref_train_config"] = (f"Tile.train_batch at cfg.yaml sizes: {n} rays (one 91x91 patch), sparse sampling "
                               f"{S} + background {NB} + reflection {RS} samples per ray, {int(tile.cells().numel())} "
                               f"of {D ** 3} dilated cells baked per diffuse step; flag 0 diffuse, 1 specular, 2 both; "
                               "samplers, forward, masked MSE, adjoints, Adam")
    return res


def operators_bench(args, dev):
    """The remaining operators at frame size: the library's own C++ frame driver (snisr_scene_* /
    snisr_graph_*: camera rays, BVH bound and MFMA render captured in one HIP graph) on the C2 frame,
    and the reference's dense FP32 marcher (render_diffuse_kernel, training/src/cuda_func.cu:
    1687-1802) on a 1280x720 view of a dense-format scene (4x4x1 tiles of 64^3 voxels, 25% of 8^3
    blocks occupied at 60%), its visited tiles from tracing_tiles."""
    import numpy as np
    import torch
    from snisr import _native as N
    from snisr import dense
    from snisr import device as D
    from snisr import fastrendering as FR
    from snisr import scene as S

    res = {}

    def timed(fn, k):
        for _ in range(2):
            fn()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(k):
            fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) * 1e3 / k

    sc, cam, mesh = S.config_c2()
    ns = D.NativeScene(sc, N.SNISR_F16)
    dm = D.DeviceMesh(mesh.vertices, mesh.faces)
    ng = D.NativeGraph(ns, cam, N.SNISR_F16, mesh=dm)
    ms = timed(ng.render, args.extra_steps)
    assert ng.stats()["overflow"] == 0
    res["native_graph_c2_ms_per_frame"] = round(ms, 3)
    res["native_graph_c2_mrays_s"] = round(cam.H * cam.W / ms / 1e3, 2)
    del ng, ns

    ds = S.make_dense_scene(3, tile_shape=(4, 4, 1), num_voxel=64, block=8, block_occupancy=0.25)
    T, H, W, K = ds.tile_ids.size, 720, 1280, 8
    eye = np.asarray(ds.scene_min, np.float64) + np.array([0.6, 0.7, 0.5]) * np.asarray(ds.tile_shape) * ds.tile_size
    look = np.asarray(ds.scene_min, np.float64) + np.array([2.5, 2.2, 0.4]) * ds.tile_size
    dcam = S.look_at_camera(eye, look, H, W, 900.0)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    d_np = S.camera_rays_np(dcam)
    dirs = t((d_np / np.linalg.norm(d_np, axis=1, keepdims=True)).astype(np.float32))
    n = dirs.shape[0]
    origin = t(dcam.origin.astype(np.float32))
    vis = torch.empty((n, K), dtype=torch.int32, device=dev)
    FR.tracing_tiles(dirs.reshape(H, W, 3), t(ds.tile_index_map), origin, ds.tile_shape, ds.scene_min,
                     np.asarray(ds.tile_shape, np.float32) * np.float32(ds.tile_size), ds.tile_size, 512,
                     vis.reshape(H, W, K))
    o = origin.expand(n, 3).contiguous()
    s2g = torch.arange(T, dtype=torch.int32, device=dev)
    vox, nodes, cen = t(ds.voxels), t(ds.nodes), t(ds.centers)
    dif = torch.empty((n, 3), dtype=torch.float32, device=dev)
    dep = torch.empty(n, dtype=torch.float32, device=dev)
    val = torch.empty(n, dtype=torch.int32, device=dev)
    step = 0.2 * ds.voxel_size
    ms = timed(lambda: dense.render_diffuse(o, dirs, vis, s2g, ds.tile_size, ds.num_voxel + 2, ds.voxel_size, step,
                                            cen, vox, nodes, dif, dep, val), args.extra_steps)
    res["dense_fp32_ms_per_frame"] = round(ms, 3)
    res["dense_fp32_mrays_s"] = round(n / ms / 1e3, 2)
    res["dense_fp32_valid_frac"] = round(float(val.float().mean()), 4)
    res["operators_config"] = ("native_graph: C2 frame through snisr_graph_render (one HIP graph: rays, BVH bound, "
                               "MFMA render); dense_fp32: render_diffuse on a 1280x720 view of a 4x4x1-tile dense "
                               "scene, 64^3 voxels per tile, step 0.2 voxel, K=8 visited tiles")
    return res


def ref_pipeline_bench(args, dev):
    """The reference's own frame pipeline (FRender.render form, rendering/src/__init__.py:247-341) at
    1280x720 through the FASTRENDERING stand-in: octree room (4x4x1 tiles, 30% of blocks occupied,
    16^3 voxels per block at 50%), 8 groups with 63-64x5-28 reflection MLPs, 4 x 16 reflection
    samples per 2x-downscaled pixel.  Includes the pipeline's own two host synchronisations."""
    import torch
    from snisr import frender
    from snisr import scene as S

    osc = S.make_octree_scene(12, tile_shape=(4, 4, 1), block_occupancy=0.3, n_groups=8)
    params, centers = S.make_reflection_groups(13, 8, (0, 0, 0), (4, 4, 1))
    cam = S.room_camera(2, (0, 0, 0), (4, 4, 1), 720, 1280)
    fr = frender.FRender(osc, params, centers, H=720, W=1280)
    fr.set_camera(cam)
    for _ in range(2):
        fr.render()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.ref_frames):
        fr.render()
    torch.cuda.synchronize()
    ms = (time.perf_counter() - t0) * 1e3 / args.ref_frames

    def graphed_ms():
        fr._graph = None
        ref = fr.render().clone()
        for _ in range(2):
            out = fr.render_graphed()
        torch.cuda.synchronize()
        assert torch.equal(out, ref)  # the replayed frame is the reference-form frame
        t = time.perf_counter()
        for _ in range(args.ref_frames):
            fr.render_graphed()
        torch.cuda.synchronize()
        return (time.perf_counter() - t) * 1e3 / args.ref_frames

    # the same frame without host synchronisation (device-side regrouping), captured in a HIP graph
    ms_graph = graphed_ms()
    # the same frame with the U-Net refinement enabled (FP16, random weights of the reference's shape)
    torch.manual_seed(0)
    fr.load_cnn()
    for _ in range(2):
        fr.render()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.ref_frames):
        fr.render()
    torch.cuda.synchronize()
    ms_cnn = (time.perf_counter() - t0) * 1e3 / args.ref_frames
    ms_cnn_graph = graphed_ms()
    psnr = {}
    if not args.no_cpu:
        # the plain frame (no U-Net: the refinement network is random here) on 600 seeded pixels
        # against the oracle chain with the reflection MLPs in FP64
        import numpy as np
        sys.path.insert(0, os.path.join(REPO, "oracle"))
        import oracle as O
        fr.cnn = None
        frame = fr.render().cpu().numpy().reshape(-1, 3)
        hi = np.sort(np.random.default_rng(31).choice(720 * 1280, 600, replace=False))
        grid_sc = S.make_scene(0, tile_shape=osc.tile_shape, tile_size=osc.tile_size, scene_min=tuple(osc.scene_min),
                               res=8, occupancy=0.0)
        grid_sc.tile_index_map = osc.tile_index_map.copy()
        ref = O.frender_subset(osc, O.OracleScene(grid_sc), params, centers, cam.origin,
                               O.compute_rays(720, 1280, cam.intrinsic, cam.c2w), 720, 1280, fr.far, hi)
        mse = float(np.mean((frame[hi].astype(np.float64) - ref["frame"]) ** 2))
        psnr["ref_pipeline_psnr_vs_fp64_db"] = round(10 * np.log10(1.0 / max(mse, 1e-30)), 2)
    return {**psnr, "ref_pipeline_ms_per_frame": round(ms, 3), "ref_pipeline_mrays_s": round(720 * 1280 / ms / 1e3, 2),
            "ref_pipeline_with_unet_ms_per_frame": round(ms_cnn, 3),
            "ref_pipeline_graphed_ms_per_frame": round(ms_graph, 3),
            "ref_pipeline_graphed_mrays_s": round(720 * 1280 / ms_graph / 1e3, 2),
            "ref_pipeline_graphed_with_unet_ms_per_frame": round(ms_cnn_graph, 3),
            "ref_pipeline_reflection_blocks": int(fr.n_reflection_blocks),
            "ref_pipeline_config": "FRender.render form at 1280x720: compute_rays, tracing_tiles (K=30), octree "
                                   "diffuse pass, sort_by_key/assign_pixels, group boundary, 4 x (inverse_z_sampling, "
                                   "inference_mlp FP16 MFMA, integrate_points) at 640x360, bilinear upsample; "
                                   "with_unet adds the 5-channel U-Net refinement in FP16; graphed: the same frame "
                                   "with the regrouping on the device (no host synchronisation), all captured in one HIP "
                                   "graph; PSNR on 600 seeded pixels of the plain frame vs the oracle chain with "
                                   "FP64 reflection MLPs; seeds 12/13/2"}


def c4_bench(args, dev):
    """C4: batched uneven tiles.  64 tiles with grids from {64,96,128}^3 and brick occupancy
    U(0.02,0.15), width-128x4 MLP in BF16 on MFMA, 4M rays with Zipf(1.2) per-tile counts, rendered
    by one launch sequence (persistent MLP kernel) captured in a HIP graph; the launch schedule is
    chosen by the autotuner."""
    import numpy as np
    import torch
    from snisr import _native as N
    from snisr import autotune
    from snisr import device as D
    from snisr import graph as G
    from snisr import scene as S

    sc, o_np, d_np, counts = S.config_c4()
    ds = D.DeviceScene(sc, mfma_dtype=N.SNISR_BF16)
    o = torch.from_numpy(o_np).to(dev)
    d = torch.from_numpy(d_np).to(dev)
    n = d.shape[0]
    ws = D.MfmaWorkspace()
    if args.c4_tuning == "auto":
        best, table = autotune.tune_render(ds, o, d, workspace=ws, reps=2)
    else:
        best, table = json.loads(args.c4_tuning), {}
    # eager (default schedule and tuned) and graph replay of the tuned schedule
    def timed(fn, k):
        fn()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(k):
            fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t0) * 1e3 / k
    out_e = D.render_mfma(ds, o, d, workspace=ws, check=True)
    eager_default = timed(lambda: D.render_mfma(ds, o, d, workspace=ws, check=False, outputs=out_e), args.c4_steps)
    eager_tuned = timed(lambda: D.render_mfma(ds, o, d, workspace=ws, check=False, tuning=best, outputs=out_e),
                        args.c4_steps)
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(7)]
    for e in ev:
        e.record()
    D.render_mfma(ds, o, d, workspace=ws, check=False, tuning=best, outputs=out_e, events=ev)
    torch.cuda.synchronize()
    stage = [ev[j].elapsed_time(ev[j + 1]) for j in range(6)]
    g = G.RenderGraph(ds, o, d, tuning=best)
    graph_ms = timed(g.replay, args.c4_steps)
    rgb = g.replay()["rgb"]
    total = int(out_e["total_samples"])
    res = {"c4_mrays_s": round(n / graph_ms / 1e3, 2), "c4_ms_per_batch": round(graph_ms, 3),
           "c4_eager_default_ms": round(eager_default, 3), "c4_eager_tuned_ms": round(eager_tuned, 3),
           "c4_rays": int(n), "c4_samples": total, "c4_tuning": best,
           "c4_stage_ms": {k: round(float(v), 3) for k, v in zip(
               ["schedule", "march", "tile_hist", "tile_scatter", "mlp_mfma", "reduce"], stage)},
           "c4_tuning_table_ms": {k: round(v, 3) for k, v in table.items()},
           "c4_config": "64 tiles (4x4x4), grids {64,96,128}^3, occupancy U(0.02,0.15), F=32 FP16, MLP 47-128x3-3 "
                        "BF16 MFMA FP32 acc, 4M rays Zipf(1.2) per tile, HIP-graph replay, seed 4"}
    if not args.no_cpu:
        sys.path.insert(0, os.path.join(REPO, "oracle"))
        import oracle as O
        idx = np.sort(np.random.default_rng(4).choice(n, 2000, replace=False))
        ref = O.render(O.OracleScene(sc), o_np, d_np, ray_index=idx, precision="f64")
        mse = float(np.mean((rgb.cpu().numpy()[idx].astype(np.float64) - ref["rgb"]) ** 2))
        res["c4_psnr_vs_fp64_db"] = round(10 * np.log10(1.0 / max(mse, 1e-30)), 2)
    return res


def c5_bench(args, dev):
    """C5: large scene.  256 tiles (16x16 floor plan) of 128^3 at 4% occupancy, F=32 FP16 features,
    per-tile width-128x4 MLP (FP16 MFMA, FP32 accumulation), 2M-triangle proxy mesh; 4 seeded
    1920x1080 views batched into one render (8.3M rays, per-ray origins).  One step = rays of the 4
    views, BVH first hit, the MFMA render; the step is captured once in a HIP graph and replayed."""
    import numpy as np
    import torch
    from snisr import _native as N
    from snisr import device as D
    from snisr import graph as G
    from snisr import scene as S

    sc, cams, mesh = S.config_c5()
    ds = D.DeviceScene(sc, mfma_dtype=N.SNISR_F16)
    dm = D.DeviceMesh(mesh.vertices, mesh.faces)
    n = len(cams) * cams[0].H * cams[0].W
    fg = G.FrameGraph(ds, dm, cams)
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(7)]
    for e in ev:
        e.record()
    fg.eager(ev)
    torch.cuda.synchronize()
    stage = [ev[j].elapsed_time(ev[j + 1]) for j in range(6)]
    fg.replay()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.c5_steps):
        fg.replay()
    torch.cuda.synchronize()
    ms = (time.perf_counter() - t0) * 1e3 / args.c5_steps
    total, over = D.mfma_stats(fg.ws.buf)
    assert over == 0
    outs, origins, rays, t_hit = fg.outputs, fg.origin, fg.rays, fg.t_hit
    flops = total * mlp_flops_per_sample(sc.mlp_in, sc.mlp_width, sc.mlp_layers)
    render_ms = float(sum(stage))
    # algorithmic gather + I/O bytes of the render (8 corners x (32 FP16 features + FP32 sigma) per
    # sample, direction in and colour out per ray) over the render's kernel time
    alg_bytes = total * 8 * (32 * 2 + 4) + n * 24
    mlp_tflops = flops / (stage[4] * 1e-3) / 1e12
    res = {"c5_mrays_s": round(n / ms / 1e3, 2), "c5_ms_per_step": round(ms, 3), "c5_rays": int(n),
           "c5_samples": int(total), "c5_msamples_s": round(total / ms / 1e3, 1),
           "c5_stage_ms": {k: round(float(v), 3) for k, v in zip(
               ["schedule", "march", "tile_hist", "tile_scatter", "mlp_mfma", "reduce"], stage)},
           "c5_mlp_tflops": round(mlp_tflops, 1),
           "c5_mfma_frac": round(mlp_tflops / MFMA_PEAK_F16_TFLOPS, 4),
           "c5_alg_gbs": round(alg_bytes / (render_ms * 1e-3) / 1e9, 1),
           "c5_hbm_frac_alg": round(alg_bytes / (render_ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
           "c5_march_gbs": round((total * (8 * 4 + 16) + n * 16) / (stage[1] * 1e-3) / 1e9, 1),
           "c5_config": "256 tiles (16x16x1) of 128^3 at 4%, F=32 FP16, MLP 47-128x3-3 FP16 MFMA FP32 acc, "
                        "2M-triangle BVH first hit, 4 seeded 1920x1080 views in one batch, HIP-graph replay, seed 5"}
    if not args.no_cpu:
        sys.path.insert(0, os.path.join(REPO, "oracle"))
        import oracle as O
        idx = np.sort(np.random.default_rng(5).choice(n, 2000, replace=False))
        ref = O.render(O.OracleScene(sc), origins.cpu().numpy(), rays.reshape(-1, 3).cpu().numpy(),
                       t_hit=t_hit.cpu().numpy(), ray_index=idx, precision="f64")
        mse = float(np.mean((outs["rgb"].cpu().numpy()[idx].astype(np.float64) - ref["rgb"]) ** 2))
        res["c5_psnr_vs_fp64_db"] = round(10 * np.log10(1.0 / max(mse, 1e-30)), 2)
    return res


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline and PSNR legs")
    ap.add_argument("--cpu-frac", type=float, default=0.3,
                    help="share of the frame's rays the CPU baseline renders (about 25 core-seconds at 0.3)")
    ap.add_argument("--fp32-frames", type=int, default=3)
    ap.add_argument("--train-steps", type=int, default=10, help="timed C3 training steps (0 = skip)")
    ap.add_argument("--ref-train-steps", type=int, default=5,
                    help="timed steps of the reference-form tile training legs (0 = skip)")
    ap.add_argument("--c4-steps", type=int, default=5, help="timed C4 batches (0 = skip)")
    ap.add_argument("--extra-steps", type=int, default=10,
                    help="timed frames of the native frame driver and the dense FP32 marcher (0 = skip)")
    ap.add_argument("--c4-tuning", default="auto",
                    help='C4 launch schedule: "auto" (autotuner) or a JSON dict, e.g. {} for the default')
    ap.add_argument("--c5-steps", type=int, default=3, help="timed C5 steps (0 = skip)")
    ap.add_argument("--ref-frames", type=int, default=10,
                    help="timed frames of the reference-format FRender pipeline (0 = skip)")
    ap.add_argument("--copy-probe", type=int, default=0,
                    help="only run a plain device copy of this many bytes (calibrates HBM byte counters)")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one MI355X: the render has no cross-GPU exchange in this build "
              "(--gpus must be 1)", file=sys.stderr)
        sys.exit(2)

    import numpy as np
    import torch
    from snisr import _native as N
    from snisr import device as D
    from snisr import graph as G
    from snisr import scene as S

    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    if args.copy_probe:
        a = torch.ones(args.copy_probe // 4, dtype=torch.float32, device=dev)
        b = torch.empty_like(a)
        for _ in range(3):
            b.copy_(a)
        torch.cuda.synchronize()
        print(json.dumps({"copy_probe_bytes": args.copy_probe, "dispatches": 3}))
        return
    sc, cam, mesh = S.config_c2()
    ds = D.DeviceScene(sc, mfma_dtype=N.SNISR_F16)
    dm = D.DeviceMesh(mesh.vertices, mesh.faces)
    H, W = cam.H, cam.W
    n_rays = H * W
    flops_per_sample = mlp_flops_per_sample(sc.mlp_in, sc.mlp_width, sc.mlp_layers)
    # the step (camera rays, BVH nearest hit, MFMA render) captured once in a HIP graph; the workspace
    # is sized from an eager render of the same view
    fg = G.FrameGraph(ds, dm, [cam])
    origin, rays_d, t_hit = fg.origin, fg.rays.reshape(-1, 3), fg.t_hit
    for _ in range(args.warmup):
        out = fg.eager()
    torch.cuda.synchronize()
    total_samples, overflow = D.mfma_stats(fg.ws.buf)
    assert overflow == 0
    eager_rgb = out["rgb"].clone()

    # per-stage kernel times from eager steps with HIP events between the stages
    ev = [[torch.cuda.Event(enable_timing=True) for _ in range(7)] for _ in range(args.steps)]
    for row in ev:
        for e in row:
            e.record()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for k in range(args.steps):
        fg.eager(ev[k])
    torch.cuda.synchronize()
    eager_ms = (time.perf_counter() - t0) * 1e3 / args.steps
    # the timed steps: graph replays
    for _ in range(max(1, args.warmup)):
        fg.replay()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for k in range(args.steps):
        fg.replay()
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    ms_per_step = (t1 - t0) * 1e3 / args.steps
    assert not fg.overflowed()
    out = fg.outputs
    assert torch.equal(out["rgb"], eager_rgb)   # the replay renders the same frame
    stage = np.array([[ev[k][j].elapsed_time(ev[k][j + 1]) for j in range(6)] for k in range(args.steps)])
    stage_ms = stage.mean(0)
    mlp_ms = float(stage_ms[4])
    mrays = n_rays / (ms_per_step * 1e-3) / 1e6

    flops = total_samples * flops_per_sample
    achieved = flops / (mlp_ms * 1e-3) / 1e12
    roofline = dict(bound="mfma", achieved=round(achieved, 2), peak=MFMA_PEAK_F16_TFLOPS, unit="TFLOP/s",
                    frac=round(achieved / MFMA_PEAK_F16_TFLOPS, 4), traffic=MLP_HBM_BYTES_PER_LAUNCH,
                    traffic_unit="bytes/launch",
                    kernel="k_mlp_mfma<32,128,4,f16 feats,f16 MFMA>",
                    flop_per_launch=flops, samples_per_launch=total_samples)
    # the traversal / compositing half on the HBM roofline: algorithmic bytes of the sigma-only march
    # (8 sigma corners x 4 B gathered and one 16 B record written per sample, direction + mesh bound
    # 16 B read per ray) and of the ordered reduction (16 B read per sample, 12 B written per ray)
    march_bytes = total_samples * (8 * 4 + 16) + n_rays * 16
    reduce_bytes = total_samples * 16 + n_rays * 12
    march_gbs = march_bytes / (float(stage_ms[1]) * 1e-3) / 1e9
    reduce_gbs = reduce_bytes / (float(stage_ms[5]) * 1e-3) / 1e9
    roofline_march = dict(bound="hbm", kernel="k_march_render", achieved=round(march_gbs, 1), peak=HBM_PEAK_GBS,
                          unit="GB/s", frac=round(march_gbs / HBM_PEAK_GBS, 4), bytes_per_launch=int(march_bytes),
                          reduce_achieved=round(reduce_gbs, 1), reduce_frac=round(reduce_gbs / HBM_PEAK_GBS, 4))

    rgb = out["rgb"].cpu().numpy()
    extra = {}
    # the FP16 MFMA rate a vendor GEMM (torch.matmul, 8192^3) sustains on the same box, beside the
    # published peak: the MLP kernel's fraction of it says how close it runs to what this part sustains
    ga = torch.randn(8192, 8192, device=dev, dtype=torch.float16)
    gb = torch.randn(8192, 8192, device=dev, dtype=torch.float16)
    for _ in range(3):
        gc = ga @ gb
    torch.cuda.synchronize()
    a = time.perf_counter()
    for _ in range(10):
        gc = ga @ gb
    torch.cuda.synchronize()
    gemm_tflops = 2 * 8192 ** 3 / ((time.perf_counter() - a) / 10) / 1e12
    del ga, gb, gc
    extra["gemm_fp16_8192_tflops"] = round(gemm_tflops, 1)
    extra["mlp_vs_gemm_fp16"] = round(achieved / gemm_tflops, 3)
    # a STREAM-style device copy (1 GiB read + 1 GiB written) beside the published 8 TB/s: the HBM
    # rate this part sustains
    src = torch.empty(1 << 28, dtype=torch.float32, device=dev).fill_(1.0)
    dst = torch.empty_like(src)
    for _ in range(3):
        dst.copy_(src)
    torch.cuda.synchronize()
    a = time.perf_counter()
    for _ in range(10):
        dst.copy_(src)
    torch.cuda.synchronize()
    copy_gbs = 2 * src.numel() * 4 / ((time.perf_counter() - a) / 10) / 1e9
    del src, dst
    extra["hbm_copy_gbs"] = round(copy_gbs, 1)
    extra["march_vs_copy_rate"] = round(march_gbs / copy_gbs, 3)
    # plain FP32 path (eight lanes per ray) on the same frame, for the MFMA/FP32 speed ratio
    if args.fp32_frames > 0:
        D.render_fp32(ds, origin, rays_d, t_hit=t_hit, image_width=W)
        torch.cuda.synchronize()
        a = time.perf_counter()
        for _ in range(args.fp32_frames):
            o32 = D.render_fp32(ds, origin, rays_d, t_hit=t_hit, image_width=W)
        torch.cuda.synchronize()
        fp32_ms = (time.perf_counter() - a) * 1e3 / args.fp32_frames
        render_ms = float(stage_ms.sum())
        extra["fp32_path_ms_per_frame"] = round(fp32_ms, 3)
        extra["mfma_vs_fp32_path_render_speedup"] = round(fp32_ms / render_ms, 2)
        extra["counts_equal_fp32_path"] = bool(torch.equal(o32["n_samples"], out["n_samples"]))

    progress("C2 headline and FP32 path done")
    if args.train_steps > 0:
        extra.update(train_bench(args, dev))
        progress("C3 training done")
    if args.ref_train_steps > 0:
        extra.update(ref_train_bench(args, dev))
        progress("reference-form training done")
    if args.ref_frames > 0:
        extra.update(ref_pipeline_bench(args, dev))
        progress("reference pipeline done")
    if args.extra_steps > 0:
        extra.update(operators_bench(args, dev))
        progress("native frame driver and dense FP32 marcher done")
    if args.c4_steps > 0:
        extra.update(c4_bench(args, dev))
        progress("C4 done")
    if args.c5_steps > 0:
        extra.update(c5_bench(args, dev))
        progress("C5 done")

    cpu = None
    if not args.no_cpu:
        dirs_np = rays_d.reshape(-1, 3).cpu().numpy()
        th_np = t_hit.cpu().numpy()
        extra["psnr_vs_fp64_db"] = round(psnr_vs_fp64(sc, cam, dirs_np, th_np, rgb), 2)
        progress("C2 PSNR vs FP64 done")
        cpu = cpu_baseline(sc, cam, dirs_np, th_np, args.cpu_frac)
        progress("CPU baseline done")

    result = {
        "metric": METRIC,
        "value": round(mrays, 2),
        "unit": "Mrays/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f16",
        "data": "synthetic",
        "config": {
            "workload": "C2 full-frame render 1280x720: 4x4x1 tiles of 128^3 voxels, 5% 8^3-brick occupancy, "
                        "F=32 FP16 features + FP32 sigma, per-tile MLP 47-128-128-128-3 (FP16 MFMA, FP32 acc), "
                        "200k-triangle proxy mesh BVH first hit bounding the march, seed 2",
            "rays": n_rays,
            "samples_per_frame": int(total_samples),
            "mesh_triangles": int(mesh.faces.shape[0]),
            "density_unit": "stored sigma = exp(N(0,1)) / voxel_size (optical depth per voxel length); "
                            "sample step 0.2 voxel; the march stops at T < 1e-3 or the mesh hit",
        },
        "msamples_s": round(total_samples / (ms_per_step * 1e-3) / 1e6, 1),
        "eager_ms_per_step": round(eager_ms, 4),
        "stage_ms": {k: round(float(v), 4) for k, v in zip(
            ["schedule", "march", "tile_hist", "tile_scatter", "mlp_mfma", "reduce"], stage_ms)},
        "roofline": roofline,
        "roofline_march": roofline_march,
        "cpu_baseline": cpu,
        **extra,
    }
    print(json.dumps(result), flush=True)


if __name__ == "__main__":
    main()
