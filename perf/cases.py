"""The work whose speed this repository tracks: what programs built on it call, over the sizes they
call it with.

Each case is one call, or one short sequence of calls, through the public Python layer: rendered
frames and ray batches, one training step of each training form, and the operators of the
reference's frame pipeline.  ``prepare`` makes the inputs and whatever a program keeps between
calls, ``run`` is one pass, ``exact`` is the same result in 64 bits written with plain torch.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch
import torch.nn.functional as F

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "scalable-neural-indoor-scene-rendering_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda"
STEP_OF = 0.2           # sample step in voxels (the renderer's sample_step_scale)
EARLY_STOP = 1e-3

# MLP shapes of the feature scenes: name -> (features, width, layers)
MLPS = {"w64": (16, 64, 3), "w128": (32, 128, 4)}


def listed():
    return [
        # a single-tile preview at 320x180: a few microseconds per kernel, so launches and ramps count
        dict(name="frame-small", kind="frame", H=180, W=320, views=1, tx=1, ty=1, res=64, occ=0.1, mlp="w64",
             dtype="f16", half=False, tris=0),
        # the interactive frame: 1280x720 in the 16-tile room, the proxy mesh bounding the march
        dict(name="frame-room", kind="frame", H=720, W=1280, views=1, tx=4, ty=4, res=128, occ=0.05, mlp="w128",
             dtype="f16", half=True, tris=200_000),
        # offline views: two 1920x1080 cameras of a floor plan in one batch
        dict(name="views-large", kind="frame", H=1080, W=1920, views=2, tx=8, ty=8, res=128, occ=0.04, mlp="w128",
             dtype="f16", half=True, tris=60_000),
        # rays of many tiles with uneven counts and grids, in random order, in BF16
        dict(name="batch-uneven", kind="batch", n=1_000_003, tx=3, ty=3, tz=3, mlp="w128", dtype="bf16"),
        # the plain FP32 path on the single-tile view
        dict(name="frame-fp32", kind="fp32", H=180, W=320, res=64, occ=0.1, mlp="w64", half=False),
        # one training step of the 16-tile room, 8192 rays per tile
        dict(name="train-room", kind="train", tx=4, ty=4, res=128, occ=0.05, rays=8192, mlp="w128"),
        # one training step on one tile with an odd, small batch
        dict(name="train-tile", kind="train", tx=1, ty=1, res=64, occ=0.1, rays=3001, mlp="w64"),
        # the tile training step's diffuse form on a 91x91 patch: bake, grid samples, background MLP
        dict(name="step-diffuse", kind="diffuse", patch=91, nv=64, samples=64, bg=32),
        # the tile training step's specular form: reflection MLP, SH head, compositing
        dict(name="step-specular", kind="specular", patch=91, samples=64),
        # the diffuse layer of the reference-format frame: rays, tile lists, octree march
        dict(name="octree-frame", kind="octree", H=720, W=1280, tx=4, ty=4),
        # the reflection layer of the same frame at half resolution: regrouping, 4 x 16 samples
        dict(name="reflection-frame", kind="reflect", H=360, W=640, groups=8),
        # the screen-space refinement network on that frame
        dict(name="refine-frame", kind="unet", H=720, W=1280),
    ]


def draw(rng):
    lg = lambda a, b: int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))  # noqa: E731
    kind = rng.choice(["frame", "batch", "fp32", "train", "diffuse", "specular", "octree", "reflect", "unet"])
    if kind == "frame":
        mlp = rng.choice(["w64", "w128", "w128"])
        n = rng.randint(1, 6)
        return dict(kind=kind, H=lg(60, 720), W=lg(80, 1280), views=rng.randint(1, 2), tx=n, ty=rng.randint(1, n),
                    res=rng.choice([64, 96, 128]), occ=round(rng.uniform(0.02, 0.12), 3), mlp=mlp,
                    dtype=rng.choice(["f16", "bf16"]) if mlp == "w128" else "f16", half=mlp == "w128",
                    tris=rng.choice([0, lg(300, 100_000)]))
    if kind == "batch":
        return dict(kind=kind, n=lg(2000, 800_000), tx=rng.randint(1, 3), ty=rng.randint(1, 3), tz=rng.randint(1, 3),
                    mlp="w128", dtype=rng.choice(["bf16", "f16"]))
    if kind == "fp32":
        return dict(kind=kind, H=lg(30, 180), W=lg(50, 320), res=rng.choice([64, 96]), occ=round(rng.uniform(0.03, 0.12), 3),
                    mlp="w64", half=rng.random() < 0.5)
    if kind == "train":
        n = rng.randint(1, 4)
        return dict(kind=kind, tx=n, ty=rng.randint(1, n), res=rng.choice([64, 96, 128]), occ=round(rng.uniform(0.03, 0.1), 3),
                    rays=lg(200, 8000), mlp=rng.choice(["w64", "w128"]))
    if kind == "diffuse":
        return dict(kind=kind, patch=rng.randint(16, 91), nv=rng.choice([32, 48, 64]), samples=rng.choice([32, 48, 64]),
                    bg=rng.choice([16, 32]))
    if kind == "specular":
        return dict(kind=kind, patch=rng.randint(8, 91), samples=rng.choice([17, 32, 64]))
    if kind == "octree":
        return dict(kind=kind, H=lg(60, 720), W=lg(100, 1280), tx=rng.randint(1, 4), ty=rng.randint(1, 4))
    if kind == "reflect":
        return dict(kind=kind, H=lg(40, 360), W=lg(60, 640), groups=lg(1, 48))
    return dict(kind=kind, H=4 * lg(15, 180), W=4 * lg(20, 320))


# ----------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _scene(seed, shape, res, occ, mlp, half):
    """A feature scene of the library's synthetic kind (``snisr.scene.make_scene``: random bricks,
    features N(0, 0.5), density e^N per voxel, Xavier MLPs), its large arrays drawn on the GPU."""
    from snisr import scene as S
    feat, width, layers = MLPS[mlp]
    rng = np.random.default_rng(seed)
    shape = np.asarray(shape, np.int32)
    T = int(shape.prod())
    cells = np.stack(np.meshgrid(*[np.arange(s) for s in shape], indexing="ij"), -1).reshape(-1, 3)
    tile_res = (np.full(T, res) if isinstance(res, int) else rng.choice(res, T)).astype(np.int32)
    p = np.full(T, occ) if isinstance(occ, float) else rng.uniform(occ[0], occ[1], T)
    counts = (tile_res // 8).astype(np.int64) ** 3
    base = np.concatenate([[0], np.cumsum(counts)[:-1]]).astype(np.int32)
    full = np.concatenate([rng.permutation(c) < max(1, round(q * c)) for c, q in zip(counts, p)])
    nb = int(full.sum())
    bmap = np.full(full.size, -1, np.int32)
    bmap[full] = np.arange(nb, dtype=np.int32)
    vs = np.repeat(1.0 / tile_res, counts)[full]
    g = _gen(seed)
    sigma = torch.exp(torch.randn((nb, 512), generator=g, device=DEV)) / torch.from_numpy(vs).to(DEV, torch.float32)[:, None]
    feats = torch.randn((nb, 512, feat), generator=g, device=DEV) * 0.5
    params = []
    for _ in range(T):
        for i, o in S.mlp_layer_dims(feat + 15, width, layers):
            a = math.sqrt(6.0 / (i + o))
            params += [rng.uniform(-a, a, i * o), np.zeros(o)]
    params = np.concatenate(params).astype(np.float32).reshape(T, -1)
    if half:
        feats, params = feats.half(), params.astype(np.float16).astype(np.float32)
    return S.Scene(tile_shape=shape, scene_min=np.zeros(3, np.float32), tile_size=1.0,
                   tile_index_map=np.arange(T, dtype=np.int32), tile_centers=(cells + 0.5).astype(np.float32),
                   tile_res=tile_res, tile_brick_base=base, brick_map=bmap, sigma=sigma.cpu().numpy(),
                   feats=feats.cpu().numpy(), mlp_in=feat + 15, mlp_width=width, mlp_layers=layers, mlp_params=params,
                   sample_step=float(np.float32(STEP_OF / tile_res.max())), early_stop=EARLY_STOP)


def _view_inputs(case, seed):
    """(scene, cameras, mesh or None) of a frame case."""
    from snisr import scene as S
    room = case.get("tx", 1) * case.get("ty", 1) > 1
    sc = _scene(seed, (case.get("tx", 1), case.get("ty", 1), 1), case["res"], case["occ"], case["mlp"], case["half"])
    hi = sc.tile_shape.astype(np.float64)
    H, W = case["H"], case["W"]
    cams = []
    for v in range(case.get("views", 1)):
        if room:
            cams.append(S.room_camera(seed * 10 + v, (0, 0, 0), hi, H, W, focal=0.586 * W))
        else:   # one tile, seen from outside
            e = np.random.default_rng(seed * 10 + v).standard_normal(3)
            cams.append(S.look_at_camera(0.5 + 2.0 * e / np.linalg.norm(e), (0.5, 0.5, 0.5), H, W, 0.866 * W))
    mesh = S.room_mesh(seed, (0, 0, 0), hi, case["tris"], avoid=cams[0].origin) if case.get("tris") else None
    return sc, cams, mesh


def _batch_inputs(case, seed):
    """Uneven tiles (grids 64..128, occupancy 2..15%) and rays towards Zipf(1.2)-distributed tiles."""
    shape = (case["tx"], case["ty"], case["tz"])
    sc = _scene(seed, shape, (64, 96, 128), (0.02, 0.15), case["mlp"], True)
    rng = np.random.default_rng(seed + 1)
    w = (rng.permutation(sc.n_tiles) + 1.0) ** -1.2
    tile = torch.from_numpy(rng.choice(sc.n_tiles, case["n"], p=w / w.sum())).to(DEV)
    return sc, *_rays_to(sc, tile, seed)


def _rays_to(sc, tile, seed):
    g = _gen(seed + 2)
    hi = torch.from_numpy(sc.tile_shape.astype(np.float32)).to(DEV)
    o = hi * torch.rand((tile.numel(), 3), generator=g, device=DEV)
    ctr = torch.from_numpy(sc.tile_centers).to(DEV)[tile]
    return o, ctr + torch.rand((tile.numel(), 3), generator=g, device=DEV) - 0.5 - o


def _train_inputs(case, seed):
    sc = _scene(seed, (case["tx"], case["ty"], 1), case["res"], case["occ"], case["mlp"], False)
    o, d = _rays_to(sc, torch.arange(sc.n_tiles, device=DEV).repeat_interleave(case["rays"]), seed)
    return sc, o, d, torch.rand((o.shape[0], 3), generator=_gen(seed + 3), device=DEV)


def _patch_inputs(case, seed):
    """A patch of rays through a tile at the origin (voxel size 0.02) with a photometric target, sorted
    depths inside the tile and background depths behind it."""
    rng = np.random.default_rng(seed)
    n, S = case["patch"] ** 2, case["samples"]
    nv = case.get("nv", 64)
    size = nv * 0.02
    o = rng.normal(size=(n, 3)) / np.sqrt(3) * 1.6 * size
    tgt = rng.uniform(-0.45, 0.45, (n, 3)) * size
    d = tgt - o
    mid = np.linalg.norm(d, axis=1, keepdims=True)
    d /= mid
    z = np.sort(np.maximum(mid + rng.uniform(-0.5, 0.5, (n, S)) * size, 0.05), axis=1)
    far = mid + size * (0.6 + np.sort(rng.uniform(0.0, 0.5, (n, case.get("bg", 1))), axis=1))
    t = lambda a: torch.tensor(a.astype(np.float32), device=DEV)  # noqa: E731
    return dict(o=t(o), d=t(d), z=t(z), bg=t(far), target=t(rng.uniform(0, 1, (n, 3))), size=size, nv=nv)


def _mlp_params(rng, depth, n_out):
    """nn.Linear order, Kaiming-uniform hidden weights, small biases."""
    out = []
    for l in range(depth):
        i, o = 63 if l == 0 else 64, n_out if l == depth - 1 else 64
        a = math.sqrt(6.0 / i) if l < depth - 1 else math.sqrt(6.0 / (i + o))
        out += [rng.uniform(-a, a, o * i), rng.normal(0.0, 0.05, o)]
    return torch.tensor(np.concatenate(out).astype(np.float32), device=DEV)


def _grid_cells(rng, nv):
    """Node flags of the dilated grid, 15% occupied."""
    D = nv + 2
    return torch.tensor(np.where(rng.uniform(0, 1, (D, D, D)) < 0.15, 1, -1).astype(np.int16), device=DEV)


def _unet_inputs(case, seed):
    """The composited frame, inverse depth and boundary flags; He-initialised weights."""
    from snisr.cnn import UNET_CONVS
    g = _gen(seed)
    H, W = case["H"], case["W"]
    low = torch.rand((1, 5, H // 4, W // 4), generator=g, device=DEV)
    x = F.interpolate(low, size=(H, W), mode="bilinear")[0]
    frame = (x[:3] + 0.05 * torch.randn((3, H, W), generator=g, device=DEV)).clamp(0, 1).permute(1, 2, 0).contiguous()
    state = {}
    for i, (ci, co) in enumerate(UNET_CONVS, start=1):
        state[f"conv{i}.weight"] = torch.randn((co, ci, 3, 3), generator=g, device=DEV) * math.sqrt(2.0 / (9 * ci)) * (0.3 if co == 3 else 1)
        state[f"conv{i}.bias"] = torch.randn(co, generator=g, device=DEV) * 0.02 + (0.4 if co == 3 else 0.0)
    return frame, x[3].contiguous(), (x[4] > 0.7)[..., None].contiguous(), state


# ----------------------------------------------------------------------------------- prepare / run
def prepare(case, seed):
    from snisr import _native as N
    from snisr import device as D
    kind = case["kind"]
    dt = {"f16": N.SNISR_F16, "bf16": N.SNISR_BF16}.get(case.get("dtype"))
    if kind == "frame":
        from snisr import graph as G
        sc, cams, mesh = _view_inputs(case, seed)
        dm = D.DeviceMesh(mesh.vertices, mesh.faces) if mesh else None
        return dict(case=case, fg=G.FrameGraph(D.DeviceScene(sc, mfma_dtype=dt), dm, cams))
    if kind == "batch":
        from snisr import graph as G
        sc, o, d = _batch_inputs(case, seed)
        return dict(case=case, g=G.RenderGraph(D.DeviceScene(sc, mfma_dtype=dt), o, d))
    if kind == "fp32":
        sc, cams, _ = _view_inputs(case, seed)
        t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
        rays = D.compute_rays(t(cams[0].intrinsic), t(cams[0].c2w), case["H"], case["W"])
        return dict(case=case, ds=D.DeviceScene(sc), o=t(cams[0].origin), d=rays.reshape(-1, 3))
    if kind == "train":
        from snisr import train as TRN
        sc, o, d, target = _train_inputs(case, seed)
        ds, ws = D.DeviceScene(sc), TRN.TrainWorkspace()
        with torch.no_grad():
            TRN.train_forward(ds, o, d, workspace=ws)   # sizes the workspace, as a program's first step does
        p = [t.clone().requires_grad_(True) for t in (ds.sigma, ds.feats, ds.mlp_params)]
        return dict(case=case, ds=ds, ws=ws, p=p, o=o, d=d, target=target)
    if kind in ("diffuse", "specular"):
        from snisr import train_ref as TR
        st = dict(case=case, **_patch_inputs(case, seed))
        rng = np.random.default_rng(seed + 1)
        depth, n_out, slope = (8, 4, 0.0) if kind == "diffuse" else (6, 28, 0.01)
        st["mlp"] = TR.PEMLP(depth, n_out, slope, device=DEV)
        with torch.no_grad():
            st["mlp"].params.copy_(_mlp_params(rng, depth, n_out))
        if kind == "diffuse":
            st["cells"] = TR.flag_cells(_grid_cells(rng, case["nv"]))
        return st
    if kind == "octree":
        from snisr import scene as S
        osc = S.make_octree_scene(seed, tile_shape=(case["tx"], case["ty"], 1), n_groups=8)
        cam = S.room_camera(seed, (0, 0, 0), osc.tile_shape, case["H"], case["W"], focal=0.586 * case["W"])
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
        return dict(case=case, osc=osc, size=torch.tensor(osc.tile_shape, dtype=torch.float32) * osc.tile_size,
                    shape=torch.tensor(osc.tile_shape, dtype=torch.int32), smin=torch.from_numpy(osc.scene_min),
                    o=t(cam.origin), intr=t(cam.intrinsic), c2w=t(cam.c2w), imap=t(osc.tile_index_map),
                    tables=[t(a) for a in (osc.group_map, osc.data_voxels, osc.block_index_map, osc.nodes_index_map,
                                           osc.nodes_sample_flag, osc.voxels_start, osc.centers)])
    if kind == "reflect":
        from snisr import fastrendering as FR
        from snisr import scene as S
        rf = S.reflection_frame(seed, 2 * case["H"], 2 * case["W"], n_groups=case["groups"])
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
        n, mb = case["H"] * case["W"], FR.regroup_max_blocks(case["H"] * case["W"], 64)
        e = lambda k, ty: torch.empty(k, dtype=ty, device=DEV)  # noqa: E731
        return dict(case=case, far=rf.far, o=t(rf.origin), rays=t(rf.rays_d), near=t(rf.inverse_near),
                    net=t(rf.net_idx).flatten(), params=t(rf.params), centers=t(rf.centers),
                    rg=(e(n, torch.int32), e(mb, torch.int16), e(mb + 1, torch.int32), e(1, torch.int32),
                        e(int(N.lib().snisr_regroup_workspace_size(n)), torch.uint8)), mb=mb)
    from snisr.cnn import HipUnet
    frame, inv, bnd, state = _unet_inputs(case, seed)
    return dict(case=case, net=HipUnet(state, device=DEV), x=(frame, inv, bnd))


def run(st):
    return _RUN[st["case"]["kind"]](st)


def _run_frame(st):
    fg = st["fg"]
    out = dict(fg.replay())
    if fg.mesh is not None:
        out.update(t_hit=fg.t_hit, tri=fg.tri)
    return out


def _run_batch(st):
    return dict(st["g"].replay())


def _run_fp32(st):
    from snisr import device as D
    return D.render_fp32(st["ds"], st["o"], st["d"], image_width=st["case"]["W"])


def _run_train(st):
    from snisr import train as TRN
    for p in st["p"]:
        p.grad = None
    rgb = TRN.render(*st["p"], st["o"], st["d"], st["ds"], workspace=st["ws"])
    torch.mean((rgb - st["target"]) ** 2).backward()
    return dict(rgb=rgb.detach(), dsigma=st["p"][0].grad, dfeats=st["p"][1].grad, dmlp=st["p"][2].grad)


def _points(st, z):
    return st["o"][:, None, :] + z[..., None] * st["d"][:, None, :]


def _gaps(z, last=1e10):
    return torch.cat([z[:, 1:] - z[:, :-1], torch.full_like(z[:, :1], last)], dim=1)[..., None]


def _run_diffuse(st):
    from snisr import train_ref as TR
    mlp, D, S = st["mlp"], st["nv"] + 2, st["case"]["samples"]
    mlp.params.grad = None
    corner = (-st["size"] / 2 - 0.02,) * 3
    bg_rgb, bg_sigma = TR.inference_diffuse(mlp, _points(st, st["bg"]), (0.0, 0.0, 0.0), 4.0)
    vox = TR.bake_voxels(mlp, st["cells"], D, corner, 0.02, (0.0, 0.0, 0.0), 4.0)
    rgb, sigma = TR.query_voxel(vox, _points(st, st["z"]), corner, 0.02)
    dists = _gaps(torch.cat([st["z"], st["bg"]], dim=1))
    c, left, _ = TR.volume_rendering(rgb, sigma, dists[:, :S].contiguous())
    c_bg, _, _ = TR.volume_rendering(bg_rgb, bg_sigma, dists[:, S:].contiguous(), left[:, -1:, :])
    pred = c + c_bg
    torch.mean((pred - st["target"]) ** 2).backward()
    return dict(pred=pred.detach(), grid=vox.detach(), dparams=mlp.params.grad)


def _run_specular(st):
    from snisr import train_ref as TR
    mlp = st["mlp"]
    mlp.params.grad = None
    raw = mlp(TR.normalize_points(_points(st, st["z"]), (0.0, 0.0, 0.0), 8.0))
    spec = TR.sh_sigmoid(raw, st["d"], 2)
    pred, _, _ = TR.volume_rendering(spec, torch.relu(raw[..., -1:]), _gaps(st["z"]))
    torch.mean((pred - st["target"]) ** 2).backward()
    return dict(pred=pred.detach(), dparams=mlp.params.grad)


def _run_octree(st):
    from snisr import fastrendering as FR
    H, W, osc = st["case"]["H"], st["case"]["W"], st["osc"]
    rays = torch.empty((H, W, 3), device=DEV)
    vis = torch.empty((H, W, 30), dtype=torch.int32, device=DEV)
    frame = torch.full((H, W, 3), -1.0, device=DEV)
    near = torch.full((H, W), 1e-8, device=DEV)
    net = torch.full((H, W), -1, dtype=torch.int16, device=DEV)
    FR.compute_rays(st["intr"], st["c2w"], 256, rays)
    FR.tracing_tiles(rays, st["imap"], st["o"], st["shape"], st["smin"], st["size"], osc.tile_size, 256, vis)
    FR.rendering_diffuse_octree_fp16(rays, vis, st["o"], *st["tables"], osc.tile_size, osc.voxel_size, osc.sample_step,
                                     osc.num_voxel, 256, 0.8, 0.01, False, frame, near, net)
    return dict(rays=rays, visited=vis, frame=frame, near=near, net=net)


def _run_reflect(st):
    from snisr import fastrendering as FR
    H, W = st["case"]["H"], st["case"]["W"]
    query, bnet, bstart, nblk, ws = st["rg"]
    FR.regroup_pixels(st["net"], 64, query, bnet, bstart, nblk, ws)
    near = st["near"]
    bound = (1.0 / (1.0 / near + st["far"]) - near) / 63
    trans = torch.ones((H, W, 1), device=DEV)
    spec = torch.zeros((H, W, 3), device=DEV)
    rays = st["rays"][::2, ::2]
    res = torch.empty((H, W, 16, 4), device=DEV)
    pts = torch.empty((H, W, 16, 3), device=DEV)
    steps = torch.empty((H, W, 16), device=DEV)
    for k in range(0, 64, 16):
        res.zero_()
        FR.inverse_z_sampling(st["o"], rays, near, bound, 256, k, 16, pts, steps)
        FR.inference_mlp(16, st["mb"], 256, 1.0 / st["far"], 0.01, bnet, trans, query, bstart, st["centers"], pts, rays,
                         st["params"], res, n_blocks_device=nblk)
        FR.integrate_points(res, steps, 512, 0.01, trans, spec)
    return dict(spec=spec, trans=trans)


def _run_unet(st):
    return dict(frame=st["net"](*st["x"]))


_RUN = dict(frame=_run_frame, batch=_run_batch, fp32=_run_fp32, train=_run_train, diffuse=_run_diffuse,
            specular=_run_specular, octree=_run_octree, reflect=_run_reflect, unet=_run_unet)


# ----------------------------------------------------------------------------------- work
def work(case):
    """Bytes and operations of one pass.  Sample counts of the marches are the means these scenes give
    (about 9 composited samples per camera ray, 25 per arbitrary ray)."""
    kind = case["kind"]
    if kind in ("frame", "fp32", "batch", "train"):
        feat, width, layers = MLPS[case["mlp"]]
        dims = [feat + 15] + [width] * (layers - 1) + [3]
        mac = sum(a * b for a, b in zip(dims, dims[1:]))
        tiles = case.get("tx", 1) * case.get("ty", 1) * case.get("tz", 1)
        occ, res = case.get("occ", 0.08), case.get("res", 96)
        vox = tiles * occ * res ** 3
        elem = 2 if case.get("half", True) and kind != "train" else 4
        n = case["n"] if kind == "batch" else tiles * case["rays"] if kind == "train" else \
            case["H"] * case["W"] * case.get("views", 1)
        s = n * (9 if kind in ("frame", "fp32") else 25)
        scene = min(vox, 8 * s) * (4 + feat * elem)
        if kind == "train":   # forward and both adjoint products; gradients of every voxel and weight
            return dict(bytes=scene + 36 * n + vox * 4 * (1 + feat) + 8 * tiles * mac, flops=6 * mac * s)
        return dict(bytes=scene + 48 * n, flops=2 * mac * s)
    if kind in ("diffuse", "specular"):
        n = case["patch"] ** 2 * case["samples"]
        if kind == "specular":
            mac = 63 * 64 + 4 * 64 * 64 + 64 * 28
            return dict(bytes=n * 4.0 + 36 * case["patch"] ** 2, flops=6 * mac * n)
        mac = 63 * 64 + 6 * 64 * 64 + 64 * 4
        cells = 0.15 * (case["nv"] + 2) ** 3
        return dict(bytes=4 * n + 16 * (case["nv"] + 2) ** 3 + 4 * cells,
                    flops=6 * mac * (cells + case["patch"] ** 2 * case["bg"]) + 120 * n)
    n = case["H"] * case["W"]
    if kind == "octree":
        return dict(bytes=n * (12 + 120 + 12 + 4 + 2) + case["tx"] * case["ty"] * 19 * 5832 * 7, flops=n * 30 * 150)
    if kind == "reflect":
        return dict(bytes=n * (12 + 4 + 2 + 16) + case["groups"] * 45112, flops=n * 64 * 2.0 * (63 * 64 + 4 * 64 * 64 + 64 * 28))
    full = 5 * 64 + 64 * 32 + 96 * 32 + 32 * 3
    half = 32 * 64 + 64 * 64 + 192 * 64 + 64 * 64
    return dict(bytes=n * (12 + 4 + 1 + 12), flops=18.0 * n * (full + half / 4 + (64 * 128 + 128 * 128) / 16))


# ----------------------------------------------------------------------------------- exact
def exact(case, seed):
    kind = case["kind"]
    if kind in ("frame", "fp32"):
        sc, cams, mesh = _view_inputs(case, seed)
        o, d = zip(*[_camera_rays(c) for c in cams])
        o, d = torch.cat(o), torch.cat(d)
        t_hit = _box_hits(mesh, o, d) if mesh else None
        rgb, T = _render64(sc, o, d, t_hit)
        out = dict(rgb=rgb, T=T, n_samples=None, depth=None)
        return dict(out, t_hit=t_hit, tri=None) if mesh else out
    if kind == "batch":
        sc, o, d = _batch_inputs(case, seed)
        rgb, T = _render64(sc, o.double(), d.double())
        return dict(rgb=rgb, T=T, n_samples=None, depth=None)
    if kind == "train":
        sc, o, d, target = _train_inputs(case, seed)
        rgb, _, grads = _render64(sc, o.double(), d.double(), target=target.double())
        return dict(rgb=rgb, dsigma=grads[0], dfeats=grads[1], dmlp=grads[2])
    if kind in ("diffuse", "specular"):
        return _patch64(case, seed)
    if kind == "reflect":
        return _reflect64(case, seed)
    if kind == "unet":
        return _unet64(case, seed)
    return None   # the octree march: which cells a sample falls in decides its value


def _t64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV, torch.float64)


def _camera_rays(cam):
    cx, cy, inv_f = (float(v) for v in cam.intrinsic)
    y, x = torch.meshgrid(torch.arange(cam.H, device=DEV, dtype=torch.float64),
                          torch.arange(cam.W, device=DEV, dtype=torch.float64), indexing="ij")
    v = torch.stack([(x - cx) * inv_f, (y - cy) * inv_f, torch.ones_like(x)], -1).reshape(-1, 3)
    d = v @ _t64(cam.c2w).reshape(3, 3).T
    return _t64(cam.origin).expand_as(d), d


def _slabs(o, inv, lo, hi):
    """Entry and exit of rays (N, 1) through boxes (1, B): [N, B] each."""
    near = far = None
    for a in range(3):
        u, v = (lo[None, :, a] - o[:, a, None]) * inv[:, a, None], (hi[None, :, a] - o[:, a, None]) * inv[:, a, None]
        l, h = torch.minimum(u, v), torch.maximum(u, v)
        near, far = (l, h) if near is None else (torch.maximum(near, l), torch.minimum(far, h))
    return near, far


def _box_hits(mesh, o, d):
    """Nearest surface of the boxes the mesh is made of (8 vertices each), along unit directions."""
    v = _t64(mesh.vertices).reshape(-1, 8, 3)
    lo, hi = v.amin(1), v.amax(1)
    inv = 1.0 / F.normalize(d, dim=1)
    t = torch.full((o.shape[0],), math.inf, device=DEV, dtype=torch.float64)
    rows = max(1, 60_000_000 // lo.shape[0])
    for r in range(0, o.shape[0], rows):
        n, f = _slabs(o[r:r + rows], inv[r:r + rows], lo, hi)
        hit = torch.where(n > 0, n, f)
        t[r:r + rows] = torch.where((f >= n) & (hit > 0), hit, math.inf).amin(1)
    return t


def _corners64(bmap, n, f):
    """Slots (or -1) and weights of the eight corners of voxel coordinates f [M, 3]; n, bmap base per row."""
    base, table = bmap
    i0 = torch.floor(f).long()
    w = f - i0
    nb = n // 8
    slots, weights = [], []
    for q in range(8):
        side = torch.tensor([q & 1, (q >> 1) & 1, q >> 2], device=DEV)
        x = i0 + side
        inside = ((x >= 0) & (x < n[:, None])).all(1)
        xb, xl = torch.where(inside[:, None], x, 0) // 8, torch.where(inside[:, None], x, 0) % 8
        b = table[base + (xb[:, 0] * nb + xb[:, 1]) * nb + xb[:, 2]]
        slots.append(torch.where(inside & (b >= 0), b * 512 + (xl[:, 0] * 8 + xl[:, 1]) * 8 + xl[:, 2], -1))
        weights.append(torch.where(side.bool(), w, 1 - w).prod(1))
    return torch.stack(slots, 1), torch.stack(weights, 1)


def _march64(sc, o, u, t_hit):
    """The composited samples of every ray, in ray order: dict of ray, order along the ray, tile, voxel
    coordinate and interval.  A ray visits the occupied bricks it crosses in order, samples each from
    its entry in sample_step, and stops after the sample that takes its transmittance below
    early_stop, or at t_hit."""
    N = o.shape[0]
    inv = 1.0 / u
    nmap = torch.from_numpy(sc.brick_map).to(DEV).long()
    sigma = _t64(sc.sigma).reshape(-1)
    ctr, res = _t64(sc.tile_centers), torch.from_numpy(sc.tile_res).to(DEV).long()
    tbase = torch.from_numpy(sc.tile_brick_base).to(DEV).long()
    pr, pn, pf, pt = [], [], [], []
    for t in range(sc.n_tiles):
        n, f = _slabs(o, inv, ctr[t:t + 1] - 0.5, ctr[t:t + 1] + 0.5)
        rays = torch.nonzero((f > n.clamp(min=0))[:, 0])[:, 0]
        nb = int(res[t]) // 8
        cell = torch.nonzero(nmap[tbase[t]:tbase[t] + nb ** 3] >= 0)[:, 0]
        if not len(rays) or not len(cell):
            continue
        lo = ctr[t] - 0.5 + torch.stack([cell // (nb * nb), cell // nb % nb, cell % nb], 1).double() / nb
        rows = max(1, 40_000_000 // len(cell))
        for r in range(0, len(rays), rows):
            k = rays[r:r + rows]
            n, f = _slabs(o[k], inv[k], lo, lo + 1.0 / nb)
            n = n.clamp(min=0)
            i, j = torch.nonzero(f > n, as_tuple=True)
            pr.append(k[i]); pn.append(n[i, j]); pf.append(f[i, j]); pt.append(torch.full_like(i, t))
    cat = lambda v, ty: torch.cat(v) if v else torch.empty(0, device=DEV, dtype=ty)  # noqa: E731
    pr, pn, pf, pt = cat(pr, torch.long), cat(pn, torch.float64), cat(pf, torch.float64), cat(pt, torch.long)
    by = torch.argsort(pn)
    by = by[torch.argsort(pr[by], stable=True)]
    pr, pn, pf, pt = pr[by], pn[by], pf[by], pt[by]
    counts = torch.bincount(pr, minlength=N)
    first = torch.cumsum(counts, 0) - counts
    T = torch.ones(N, device=DEV, dtype=torch.float64)
    done = torch.zeros(N, device=DEV, dtype=torch.bool)
    order = torch.zeros(N, device=DEV, dtype=torch.long)
    step = sc.sample_step
    out = [[] for _ in range(5)]
    for j in range(int(counts.max()) if len(pr) else 0):
        ray = torch.nonzero((counts > j) & ~done)[:, 0]
        at = first[ray] + j
        k = 0
        while len(ray):
            t = pn[at] + k * step
            live = (t < pf[at]) & ~done[ray]
            if t_hit is not None:
                stop = live & (t >= t_hit[ray])
                done[ray[stop]] = True
                live = live & ~stop
            ray, at, t = ray[live], at[live], t[live]
            tile = pt[at]
            f = (o[ray] + t[:, None] * u[ray] - ctr[tile] + 0.5) * res[tile, None] - 0.5
            slot, w = _corners64((tbase[tile], nmap), res[tile], f)
            s = (torch.where(slot >= 0, sigma[slot.clamp(min=0)], 0.0) * w).sum(1)
            dt = torch.minimum(torch.full_like(t, step), pf[at] - t)
            for v, x in zip(out, (ray, order[ray], tile, f, dt)):
                v.append(x)
            T[ray] = T[ray] * torch.exp(-s * dt)
            order[ray] += 1
            done[ray] = T[ray] < sc.early_stop
            k += 1
    ray, pos, tile, f, dt = (torch.cat(v) if v else None for v in out)
    return None if ray is None else dict(ray=ray, pos=pos, tile=tile, f=f, dt=dt, tbase=tbase, nmap=nmap, res=res,
                                         sigma=sigma, longest=int(order.max()))


def _render64(sc, o, d, t_hit=None, target=None):
    """(rgb, T) of the rays, and with a target the gradients of mean((rgb - target)^2) with respect to
    density, features and MLP parameters."""
    N = o.shape[0]
    u = F.normalize(d, dim=1)
    rgb, T = torch.zeros((N, 3), device=DEV, dtype=torch.float64), torch.ones(N, device=DEV, dtype=torch.float64)
    feats = torch.from_numpy(sc.feats.reshape(-1, sc.feat_dim)).to(DEV)
    params = _t64(sc.mlp_params)
    g = [torch.zeros((sc.n_bricks, 512), device=DEV, dtype=torch.float64),
         torch.zeros((sc.n_bricks, 512, sc.feat_dim), device=DEV, dtype=torch.float64), torch.zeros_like(params)] \
        if target is not None else None
    rows = 400_000
    for r in range(0, N, rows):
        part = slice(r, r + rows)
        m = _march64(sc, o[part], u[part], None if t_hit is None else t_hit[part])
        if m is None:
            continue
        n = o[part].shape[0]
        M = len(m["ray"])
        slot, w, s = [torch.empty((M, 8), device=DEV, dtype=ty) for ty in (torch.long, torch.float64)] + [None]
        for k in range(0, M, 2_000_000):
            q = slice(k, k + 2_000_000)
            slot[q], w[q] = _corners64((m["tbase"][m["tile"][q]], m["nmap"]), m["res"][m["tile"][q]], m["f"][q])
        s = (torch.where(slot >= 0, m["sigma"][slot.clamp(min=0)], 0.0) * w).sum(1).requires_grad_(g is not None)
        enc = [u[part]] + [fn(k * u[part]) for k in (1.0, 2.0) for fn in (torch.sin, torch.cos)]
        enc = torch.cat(enc, 1)

        def colours(k, grad=None):
            x = torch.zeros((len(k), sc.feat_dim), device=DEV, dtype=torch.float64)
            for c in range(8):
                x += feats[slot[k, c].clamp(min=0)].double() * (w[k, c] * (slot[k, c] >= 0))[:, None]
            x = x.requires_grad_(grad is not None)
            P = params[t].clone().requires_grad_(grad is not None)
            h, at = torch.cat([x, enc[m["ray"][k]]], 1), 0
            for l in range(sc.mlp_layers):
                i, q = h.shape[1], 3 if l == sc.mlp_layers - 1 else sc.mlp_width
                h = h @ P[at:at + i * q].reshape(q, i).T + P[at + i * q:at + i * q + q]
                at += i * q + q
                h = torch.sigmoid(h) if q == 3 else torch.relu(h)
            if grad is None:
                return h
            dx, dP = torch.autograd.grad(h, (x, P), grad)
            g[2][t] += dP
            flat = g[1].reshape(-1, sc.feat_dim)
            for c in range(8):
                use = slot[k, c] >= 0
                flat.index_add_(0, slot[k, c][use], (dx * w[k, c, None])[use])

        by_tile = [torch.nonzero(m["tile"] == t)[:, 0] for t in range(sc.n_tiles)]
        col = torch.zeros((M, 3), device=DEV, dtype=torch.float64)
        for t in range(sc.n_tiles):
            for k in by_tile[t].split(500_000):
                col[k] = colours(k)
        col.requires_grad_(g is not None)
        flat = m["ray"] * m["longest"] + m["pos"]
        tau = torch.zeros(n * m["longest"], device=DEV, dtype=torch.float64).index_put((flat,), torch.relu(s) * m["dt"])
        tau = tau.reshape(n, m["longest"])
        before = torch.exp(-(torch.cumsum(tau, 1) - tau)).reshape(-1)[flat]
        wgt = (1 - torch.exp(-torch.relu(s) * m["dt"])) * before
        out = torch.zeros((n, 3), device=DEV, dtype=torch.float64).index_add(0, m["ray"], wgt[:, None] * col)
        rgb[part], T[part] = out.detach(), torch.exp(-tau.sum(1)).detach()
        if g is not None:
            loss = ((out - target[part]) ** 2).sum() / target.numel()
            ds, dc = torch.autograd.grad(loss, (s, col))
            for c in range(8):
                use = slot[:, c] >= 0
                g[0].reshape(-1).index_add_(0, slot[use, c], (ds * w[:, c])[use])
            for t in range(sc.n_tiles):
                for k in by_tile[t].split(500_000):
                    colours(k, dc[k])
    return (rgb, T) if g is None else (rgb, T, g)


def _pe64(x):
    out = [x]
    for k in range(10):
        out += [torch.sin(2.0 ** k * x), torch.cos(2.0 ** k * x)]
    return torch.cat(out, -1)


def _mlp64(P, x, depth, n_out, slope):
    h, at = _pe64(x), 0
    for l in range(depth):
        i, o = h.shape[-1], n_out if l == depth - 1 else 64
        h = h @ P[at:at + i * o].reshape(o, i).T + P[at + i * o:at + i * o + o]
        at += i * o + o
        if l < depth - 1:
            h = F.leaky_relu(h, slope)
    return h


def _composite64(rgb, sigma, dists, T0=1.0):
    alpha = 1 - torch.exp(-sigma * dists)
    keep = torch.cumprod(1 - alpha + 1e-10, 1)
    T = torch.cat([torch.ones_like(keep[:, :1]), keep[:, :-1]], 1) * T0
    return (alpha * T * rgb).sum(1), T


def _sh64(d):
    x, y, z = d.unbind(-1)
    c = [0.28209479177387814, 0.4886025119029199, 1.0925484305920792, 0.31539156525252005, 0.5462742152960396]
    return torch.stack([torch.full_like(x, c[0]), -c[1] * y, c[1] * z, -c[1] * x, c[2] * x * y, -c[2] * y * z,
                        c[3] * (2 * z * z - x * x - y * y), -c[2] * x * z, c[4] * (x * x - y * y)], -1)


def _patch64(case, seed):
    st = {k: v.double() if isinstance(v, torch.Tensor) else v for k, v in _patch_inputs(case, seed).items()}
    rng = np.random.default_rng(seed + 1)
    pts = lambda z: st["o"][:, None, :] + z[..., None] * st["d"][:, None, :]  # noqa: E731
    if case["kind"] == "specular":
        P = _mlp_params(rng, 6, 28).double().requires_grad_(True)
        raw = _mlp64(P, pts(st["z"]) / 8.0, 6, 28, 0.01)
        Y = _sh64(F.normalize(st["d"], dim=1))[:, None, :, None]
        spec = torch.sigmoid((raw[..., :27].reshape(*raw.shape[:-1], 9, 3) * Y).sum(-2))
        pred, _ = _composite64(spec, torch.relu(raw[..., -1:]), _gaps(st["z"]))
        grid = None
    else:
        P = _mlp_params(rng, 8, 4).double().requires_grad_(True)
        cells = torch.nonzero(_grid_cells(rng, case["nv"]).reshape(-1) != -1)[:, 0]
        D, S = case["nv"] + 2, case["samples"]
        head = lambda r: torch.cat([torch.sigmoid(r[..., :3]), torch.relu(r[..., 3:])], -1)  # noqa: E731
        bg = head(_mlp64(P, pts(st["bg"]) / 4.0, 8, 4, 0.0))
        zyx = torch.stack([cells // (D * D), cells // D % D, cells % D], 1).double()
        corner = -st["size"] / 2 - 0.02
        grid = torch.zeros((D ** 3, 4), device=DEV, dtype=torch.float64)
        grid = grid.index_put((cells,), head(_mlp64(P, ((zyx.flip(1) + 0.5) * 0.02 + corner) / 4.0, 8, 4, 0.0)))
        at = ((pts(st["z"]) - corner) / 0.02 - 0.5) / (D - 1) * 2 - 1
        v = F.grid_sample(grid.reshape(1, D, D, D, 4).permute(0, 4, 1, 2, 3), at[None, None], align_corners=True)
        v = v[0, :, 0].permute(1, 2, 0)
        dists = _gaps(torch.cat([st["z"], st["bg"]], 1))
        c, T = _composite64(v[..., :3], v[..., 3:], dists[:, :S])
        pred = c + _composite64(bg[..., :3], bg[..., 3:], dists[:, S:], T[:, -1:])[0]
        grid = grid.detach().reshape(D, D, D, 4)
    (dP,) = torch.autograd.grad(((pred - st["target"]) ** 2).mean(), P)
    out = dict(pred=pred.detach(), dparams=dP)
    return out if grid is None else dict(out, grid=grid)


def _reflect64(case, seed):
    from snisr import scene as S
    rf = S.reflection_frame(seed, 2 * case["H"], 2 * case["W"], n_groups=case["groups"])
    n = case["H"] * case["W"]
    near, net = _t64(rf.inverse_near).reshape(-1, 1), torch.from_numpy(rf.net_idx.astype(np.int64)).to(DEV).reshape(-1)
    d = _t64(rf.rays_d[::2, ::2]).reshape(-1, 3)
    bound = (1 / (1 / near + rf.far) - near) / 63
    k = torch.arange(65, device=DEV, dtype=torch.float64)
    z = 1 / (bound * k + near)
    steps = (z[:, 1:] - z[:, :-1]).clamp(min=0)
    Y = _sh64(F.normalize(d, dim=1))
    P = _t64(rf.params).reshape(case["groups"], -1)
    res = torch.zeros((n, 64, 4), device=DEV, dtype=torch.float64)
    for g in range(case["groups"]):
        for p in torch.nonzero(net == g)[:, 0].split(20_000):
            x = (_t64(rf.origin) + z[p, :64, None] * d[p, None, :] - _t64(rf.centers)[g]) / rf.far
            h, at = _pe64(x), 0
            for l, (i, o) in enumerate(S.REF_MLP_DIMS):
                h = h @ P[g, at + o:at + o + i * o].reshape(i, o) + P[g, at:at + o]
                at += o + i * o
                h = F.leaky_relu(h, 0.01) if l < 5 else h
            res[p, :, :3] = torch.sigmoid((h[..., :27].reshape(*h.shape[:-1], 9, 3) * Y[p, None, :, None]).sum(-2))
            res[p, :, 3] = torch.relu(h[..., 27])
    spec = torch.zeros((n, 3), device=DEV, dtype=torch.float64)
    T = torch.ones((n, 1), device=DEV, dtype=torch.float64)
    for r in range(0, 64, 16):   # a pixel whose transmittance is below 0.01 takes no further round
        live = (T >= 0.01).double()
        for j in range(r, r + 16):
            a = (1 - torch.exp(-res[:, j, 3:] * steps[:, j:j + 1])) * live
            spec = spec + a * T * res[:, j, :3]
            T = T * (1 - a)
    return dict(spec=spec.reshape(case["H"], case["W"], 3), trans=T.reshape(case["H"], case["W"], 1))


def _unet64(case, seed):
    frame, inv, bnd, state = _unet_inputs(case, seed)
    x = torch.cat([frame.permute(2, 0, 1), inv[None], bnd.permute(2, 0, 1).float()]).double()

    def conv(i, x):
        w, b = state[f"conv{i}.weight"].double(), state[f"conv{i}.bias"].double()
        H, W = x.shape[1:]
        p = F.pad(x, (1, 1, 1, 1))
        y = b[:, None] + sum(w[:, :, t // 3, t % 3] @ p[:, t // 3:t // 3 + H, t % 3:t % 3 + W].reshape(x.shape[0], -1)
                             for t in range(9))
        return torch.relu(y).reshape(-1, H, W)

    down = lambda v: v.reshape(v.shape[0], v.shape[1] // 2, 2, v.shape[2] // 2, 2).mean((2, 4))  # noqa: E731
    up = lambda v: F.interpolate(v[None], scale_factor=2, mode="bilinear", align_corners=True)[0]  # noqa: E731
    o2 = conv(2, conv(1, x))
    o5 = conv(4, conv(3, down(o2)))
    e7 = conv(6, conv(5, down(o5)))
    e4 = conv(8, conv(7, torch.cat([up(e7), o5])))
    y = conv(10, conv(9, torch.cat([up(e4), o2])))
    return dict(frame=y.clamp(max=1.0).permute(1, 2, 0).contiguous())
