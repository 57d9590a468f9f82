"""The grid-sample adjoint where many samples share a voxel: runs shorter than, as long as and longer than the
eight-sample segments and the wavefronts that sum them, against the oracle."""
import numpy as np
import pytest
import torch

from snisr import train_ref as TR

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


# sums of n random terms in FP32, at most n / 8 of them by atomics: about 2^-24 sqrt(n / 8) of the result < 1e-5
@pytest.mark.parametrize("run", [1, 3, 8, 9, 64, 65, 20000])
@pytest.mark.parametrize("n", [1, 63, 65, 511, 20000])
def test_shared_voxels_match_oracle(oracle_mod, n, run):
    rng = np.random.default_rng(n + run)
    D, vs = 9, 0.07
    mc = np.array([-0.3, 0.2, 1.1], np.float32)
    cell = rng.integers(0, D - 1, (n // run + 1, 3)).repeat(run, 0)[:n]      # one voxel per run
    pts = (mc + (cell + rng.uniform(0.05, 0.95, (n, 3))) * vs).astype(np.float32)
    g_rgb, g_sig = rng.normal(size=(n, 3)).astype(np.float32), rng.normal(size=(n, 1)).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(DEV)  # noqa: E731
    vox = torch.zeros((D, D, D, 4), device=DEV, requires_grad=True)
    rgb, sig = TR.query_voxel(vox, t(pts), mc, vs)
    torch.autograd.backward([rgb, sig], [t(g_rgb), t(g_sig)])
    ref = oracle_mod.voxel_query(np.zeros((D, D, D, 4), np.float32), pts, mc, vs, g_rgb=g_rgb, g_sigma=g_sig)["g_vox"]
    got = vox.grad.cpu().numpy().astype(np.float64)
    assert np.linalg.norm(got - ref) <= 1e-5 * np.linalg.norm(ref)
