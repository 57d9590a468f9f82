"""The octree march reads its voxels as FP16 operands: subnormal, negative and largest halves against the FP32
oracle, the pixels within 1e-4 of their largest magnitude (the bound of the unit-scale scenes)."""
import numpy as np
import pytest

from snisr import scene as S
from test_gpu_octree import render_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [2e-6, -3e-5, 500.0])
def test_half_range_matches_oracle(oracle_mod, scale):
    def field(t, ijk):
        v = np.empty(ijk.shape[:-1] + (4,), np.float32)
        v[..., :3] = (ijk + 0.5) * np.float32(scale)
        v[..., 3] = 40.0 * (ijk.sum(-1) % 3)
        return v
    osc = S.make_octree_scene(8, tile_shape=(2, 1, 1), block_occupancy=0.6, field=field, flag_border=True)
    cam = S.look_at_camera((-1.5, 0.5, 0.6), (1.0, 0.5, 0.5), 56, 88, 60.0)
    (f, i, n, s), (rf, ri, rn, rs) = render_both(oracle_mod, osc, cam, K=4)
    assert np.array_equal(s, rs) and np.array_equal(n, rn) and s.sum() > 1000
    assert np.array_equal(i.view(np.uint32), ri.view(np.uint32))
    assert np.abs(f - rf).max() <= 1e-4 * np.abs(rf).max()
