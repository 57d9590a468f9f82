"""Batches large enough for the ray queue (more than 1536 rays per CU): counts, T and depth equal to the plain
path's bit for bit, pixels within the FP16 layers' bound, for unrelated rays (lanes fill their staged records at
different times), for one ray repeated (all at once) and for rays that all miss."""
import numpy as np
import pytest
import torch

from snisr import _native as N
from snisr import device as D
from snisr import scene as S

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("kind", ["random", "same", "miss"])
@pytest.mark.parametrize("extra", [1, 77])
def test_ray_queue_matches_plain_path(kind, extra):
    print(f"ray queue {kind} +{extra}", flush=True)
    n = 1536 * torch.cuda.get_device_properties(0).multi_processor_count + extra
    sc = S.make_scene(31, tile_shape=(3, 2, 2), res_choices=(16, 24, 64), occupancy=0.3, sample_step=1.0 / 160,
                      feat_half=False, feat_dim=16, mlp_width=64, mlp_layers=3)
    ds = D.DeviceScene(sc, mfma_dtype=N.SNISR_F16)
    rng = np.random.default_rng(extra)
    o = rng.uniform(-0.5, 3.0, (n, 3)).astype(np.float32)
    d = rng.standard_normal((n, 3)).astype(np.float32)
    if kind == "same":
        o[:], d[:] = (-0.5, 0.9, 1.1), (1.0, 0.21, -0.13)
    if kind == "miss":
        o[:, 0], d[:, 0] = -1.0, -np.abs(d[:, 0])
    o, d = torch.from_numpy(o).to(DEV), torch.from_numpy(d).to(DEV)
    ref = D.render_fp32(ds, o, d, brick_cap=4)
    out = D.render_mfma(ds, o, d, brick_cap=4)
    for k in ("n_samples", "T", "depth", "bricks"):
        assert torch.equal(out[k].view(torch.int32), ref[k].view(torch.int32)), k
    assert (out["rgb"] - ref["rgb"]).abs().max() <= 5e-3   # FP16 layers
    assert (int(ref["n_samples"].max()) > 0) == (kind != "miss")
