"""The marches that large launches take, one ray per lane: the packet march (camera frames of more than 1024 rays
per CU) and the ray queue (other batches of more than 1536), with record slots that overflow or are no multiple
of eight, march bounds and visit lists, ray orders, chunks and graph replays.  Counts, T, depth and bricks equal
those of the nested per-ray march (k_march_sigma) bit for bit; small launches take the grouped march instead."""
import numpy as np
import pytest
import torch

from snisr import _native as N
from snisr import device as D
from snisr import graph as G
from snisr import scene as S

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
MARCHED = ("n_samples", "T", "depth")


def per_cu(k):
    return k * torch.cuda.get_device_properties(0).multi_processor_count


@pytest.fixture(scope="module")
def scene():
    return S.make_scene(31, tile_shape=(3, 2, 2), res_choices=(16, 24, 32), occupancy=0.3, sample_step=1.0 / 64,
                      feat_half=False, feat_dim=16, mlp_width=64, mlp_layers=3)


@pytest.fixture(scope="module")
def ds(scene):
    return D.DeviceScene(scene, mfma_dtype=N.SNISR_F16)


def rays(kind, times=1, seed=5):
    """(origin(s), directions, image width) of more rays than the small marches take, `times` over"""
    rng = np.random.default_rng(seed)
    if kind == "queue":
        n = times * (per_cu(1536) + 77)
        o = torch.from_numpy(rng.uniform(-0.5, 3.0, (n, 3)).astype(np.float32))
        d = torch.from_numpy(rng.standard_normal((n, 3)).astype(np.float32))
        return o.to(DEV), d.to(DEV), 0
    W = 640
    H = 8 * (times * per_cu(1024) // (8 * W) + times)
    cam = S.room_camera(3, (0, 0, 0), (3, 2, 2), H, W, focal=0.6 * W)
    return torch.from_numpy(cam.origin).to(DEV), torch.from_numpy(S.camera_rays_np(cam)).to(DEV).reshape(-1, 3), W


def equal(a, b, keys):
    for k in keys:
        assert torch.equal(a[k].view(torch.int32), b[k].view(torch.int32)), k


@pytest.fixture(scope="module", params=["queue", "packets"])
def case(request, ds):
    o, d, W = rays(request.param)
    ref = D.render_mfma(ds, o, d, image_width=W)
    equal(ref, D.render_fp32(ds, o, d, image_width=W, rgb=False), MARCHED)
    assert int(ref["n_samples"].max()) > 13               # the largest slot count that overflows below
    return request.param, o, d, W, ref


def test_bounds_visit_lists_and_bricks_match_nested_march(case, scene, ds, oracle_mod):
    kind, o, d, W, _ = case
    o = o[:3].mean(0) if kind == "queue" else o            # visit lists are traced from one origin
    n = d.shape[0]
    th = torch.from_numpy(np.random.default_rng(3).uniform(0.05, 3.0, n).astype(np.float32)).to(DEV)
    th[::11] = float("inf")
    vis = D.trace_tiles(ds, o, d / d.norm(dim=1, keepdim=True), scene.max_tiles)
    for kw in (dict(t_hit=th), dict(t_hit=th, visited=vis)):
        out = D.render_mfma(ds, o, d, image_width=W, brick_cap=12, **kw)
        nested = D.render_fp32(ds, o, d, image_width=W, brick_cap=12, rgb=False, **kw)
        equal(out, nested, MARCHED + ("bricks",))
        assert (out["rgb"] - D.render_fp32(ds, o, d, image_width=W, **kw)["rgb"]).abs().max() <= 5e-3  # FP16 layers
    idx = np.sort(np.random.default_rng(0).choice(n, 2000, replace=False))
    ref = oracle_mod.render(oracle_mod.OracleScene(scene), o.cpu().numpy(), d.cpu().numpy(), t_hit=th.cpu().numpy(),
                            ray_index=idx)
    assert np.array_equal(out["n_samples"].cpu().numpy()[idx], ref["n_samples"])
    assert np.array_equal(out["T"].cpu().numpy()[idx].view(np.uint32), ref["T"].view(np.uint32))


@pytest.mark.parametrize("slots", [2, 8, 13])
def test_record_overflow_is_confined_and_recovered(case, ds, slots):
    _, o, d, W, ref = case
    ws = D.MfmaWorkspace()
    out = D.render_mfma(ds, o, d, image_width=W, workspace=ws, capacity=slots, check=False)
    total, over, most = D.mfma_stats(ws.buf, with_max=True)
    assert over == 1 and most == int(ref["n_samples"].max()) and total == int(ref["n_samples"].sum())
    equal(out, ref, MARCHED)
    fits = ref["n_samples"] <= slots
    assert torch.isnan(out["rgb"][~fits]).all() and torch.equal(out["rgb"][fits], ref["rgb"][fits])
    again = D.render_mfma(ds, o, d, image_width=W, workspace=ws, capacity=slots, check=True)
    assert torch.equal(again["rgb"], ref["rgb"])


def test_sample_overflow_skips_the_frame(case, ds):
    _, o, d, W, ref = case
    ws = D.MfmaWorkspace()
    out = D.render_mfma(ds, o, d, image_width=W, workspace=ws, capacity=128, sample_capacity=1000, check=False)
    assert D.mfma_stats(ws.buf) == (int(ref["n_samples"].sum()), 1)
    equal(out, ref, MARCHED)
    assert torch.isnan(out["rgb"]).all()


@pytest.mark.parametrize("order", [1, 2, 3])
def test_ray_orders_give_the_same_render(case, ds, order):
    _, o, d, W, ref = case
    # an order takes frames off the packet march: enough rays for the queue
    if W:
        o, d, W = rays("packets", 2)
        ref = D.render_mfma(ds, o, d, image_width=W)
    out = D.render_mfma(ds, o, d, image_width=W, tuning=dict(ray_order=order))
    equal(out, ref, MARCHED + ("rgb",))


@pytest.mark.parametrize("kind", ["queue", "packets"])
def test_chunks_of_large_marches_equal_one_pass(ds, kind):
    o, d, W = rays(kind, 2)
    ref = D.render_mfma(ds, o, d, image_width=W)
    for slots in (0, 13):
        ws = D.MfmaWorkspace()
        out = D.render_mfma(ds, o, d, image_width=W, workspace=ws, capacity=slots, check=slots == 0, tuning=dict(chunks=2))
        equal(out, ref, MARCHED)
        fits = ref["n_samples"] <= (slots or 1 << 30)
        assert torch.equal(out["rgb"][fits], ref["rgb"][fits]) and torch.isnan(out["rgb"][~fits]).all()


@pytest.mark.parametrize("tuning", [None, dict(ray_order=1), dict(chunks=2)])
def test_graph_replays_of_large_marches_match_eager(case, ds, tuning):
    kind, o, d, W, ref = case
    if tuning and "chunks" in tuning:      # each chunk above the small marches
        o, d, W = rays(kind, 2)
        ref = D.render_mfma(ds, o, d, image_width=W)
    g = G.RenderGraph(ds, o, d, image_width=W, tuning=tuning)
    for _ in range(3):
        out = g.replay()
        torch.cuda.synchronize()
        equal(out, ref, MARCHED + ("rgb",))
        torch.randn(1 << 20, device=DEV).mul_(2)
        torch.cuda.synchronize()
    assert not g.overflowed()
