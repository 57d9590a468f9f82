"""Rays marched by groups of lanes: ray counts around the wavefront and group sizes, rays of many tiles in
one wavefront, march bounds and visit lists, against the oracle (bit-exact counts, T, depth and bricks)."""
import numpy as np
import pytest
import torch

from snisr import device as D
from snisr import scene as S

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
RGB_TOL = 1e-4  # FP32 pixels vs the FP32 oracle (max abs error)


def scene(width):
    kw = dict(feat_dim=32, mlp_width=128, mlp_layers=4) if width == 128 else dict(feat_dim=16, mlp_width=width, mlp_layers=3)
    return S.make_scene(31, tile_shape=(3, 2, 2), res_choices=(16, 24, 64), occupancy=0.3, sample_step=1.0 / 160,
                        feat_half=width == 128, **kw)


def rays(n, seed):
    rng = np.random.default_rng(seed)
    o = rng.uniform(-0.5, 3.0, (n, 3)).astype(np.float32)
    d = rng.standard_normal((n, 3)).astype(np.float32)
    d[::5, 1:] = 0.0                      # axis-parallel
    return o, d, rng.uniform(0.05, 3.0, n).astype(np.float32)


@pytest.mark.parametrize("width", [32, 64, 128])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 65, 517])
def test_fp32_render_matches_oracle(oracle_mod, width, n):
    sc = scene(width)
    ds, osc = D.DeviceScene(sc), oracle_mod.OracleScene(sc)
    o, d, th = rays(n, n + width)
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    for hit in (None, th):
        out = D.render_fp32(ds, t(o), t(d), t_hit=None if hit is None else t(hit), brick_cap=24)
        ref = oracle_mod.render(osc, o, d, t_hit=hit, brick_debug=24)
        g = {k: v.cpu().numpy() for k, v in out.items()}
        for k in ("n_samples", "bricks"):
            assert np.array_equal(g[k], ref[k]), k
        for k in ("T", "depth"):
            assert np.array_equal(g[k].view(np.uint32), ref[k].view(np.uint32)), k
        assert np.abs(g["rgb"] - ref["rgb"]).max() <= RGB_TOL


# batches on either side of the group sizes: 8 lanes per ray up to 64 rays per CU, 4 up to 192, then 2; training
# 8 up to 144, then 4
@pytest.mark.parametrize("n", [1, 9, 64, 16384, 16391, 36864, 36871, 49152, 49159, 57344, 57351])
def test_small_batches_match_fp32_path(n):
    from snisr import _native as N
    from snisr import train as TRN
    sc = scene(64)
    ds = D.DeviceScene(sc, mfma_dtype=N.SNISR_F16)
    o, d, th = rays(n, n)
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    for hit in (None, t(th)):
        ref = D.render_fp32(ds, t(o), t(d), t_hit=hit, brick_cap=24)
        out = D.render_mfma(ds, t(o), t(d), t_hit=hit, brick_cap=24)
        for k in ("n_samples", "T", "depth", "bricks"):
            assert torch.equal(out[k].view(torch.int32), ref[k].view(torch.int32)), k
        assert (out["rgb"] - ref["rgb"]).abs().max() <= 5e-3   # FP16 layers
        trn, _ = TRN.train_forward(ds, t(o), t(d), t_hit=hit)
        for k in ("n_samples", "T", "depth"):
            assert torch.equal(trn[k].view(torch.int32), ref[k].view(torch.int32)), k
        assert (trn["rgb"] - ref["rgb"]).abs().max() <= 2e-5


@pytest.mark.parametrize("H,W", [(8, 8), (64, 96), (60, 96), (248, 232)])
def test_small_frames_match_fp32_path(H, W):
    from snisr import _native as N
    sc = scene(64)
    ds = D.DeviceScene(sc, mfma_dtype=N.SNISR_F16)
    cam = S.room_camera(3, (0, 0, 0), (3, 2, 2), H, W, focal=0.6 * W)
    d = torch.from_numpy(S.camera_rays_np(cam)).to(DEV)
    o = torch.from_numpy(cam.origin).to(DEV)
    ref = D.render_fp32(ds, o, d, image_width=W)
    out = D.render_mfma(ds, o, d, image_width=W)
    for k in ("n_samples", "T", "depth"):
        assert torch.equal(out[k].view(torch.int32), ref[k].view(torch.int32)), k
    assert (out["rgb"] - ref["rgb"]).abs().max() <= 5e-3
