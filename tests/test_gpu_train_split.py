"""Training MLP products: sample counts around the wavefront and workgroup sizes, operand
ranges far from one, and encoding arguments on both sides of the range-reduction limit."""
import pytest
import torch

from snisr import train_ref as TR

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def params(depth, n_out, seed):
    g = torch.Generator().manual_seed(seed)
    out = []
    for l in range(depth):
        i, o = 63 if l == 0 else 64, n_out if l == depth - 1 else 64
        out += [(torch.rand((o, i), generator=g) * 2 - 1) * (6.0 / i) ** 0.5, torch.randn(o, generator=g) * 0.05]
    return out


def forward64(p, x, slope):
    x = x.double()
    h = torch.cat([x] + [f((2.0 ** k) * x) for k in range(10) for f in (torch.sin, torch.cos)], 1)
    for l in range(0, len(p), 2):
        h = h @ p[l].double().T + p[l + 1].double()
        if l + 2 < len(p):
            h = torch.nn.functional.leaky_relu(h, slope)
    return h


def mlp(p, depth, n_out, slope):
    m = TR.PEMLP(depth, n_out, slope, device=DEV)
    with torch.no_grad():
        m.params.copy_(torch.cat([t.reshape(-1) for t in p]))
    return m


# FP32 sums over 64 inputs per layer: outputs within 1e-5 of a row's largest
@pytest.mark.parametrize("depth,n_out,slope", [(2, 4, 0.0), (6, 28, 0.01), (8, 4, 0.0)])
@pytest.mark.parametrize("n", [1, 31, 33, 127, 129, 1000])
def test_ragged_counts_match_fp64(depth, n_out, slope, n):
    p = params(depth, n_out, n + depth)
    x = torch.rand((n, 3), generator=torch.Generator().manual_seed(n)) * 2 - 1
    m = mlp(p, depth, n_out, slope)
    out = m(x.to(DEV))
    ref = forward64(p, x, slope)
    err = (out.detach().cpu().double() - ref).abs().amax(1)
    assert (err <= 1e-5 * ref.abs().amax(1).clamp(min=1.0)).all(), err.max()
    out.backward(torch.ones_like(out))
    q = [t.clone().double().requires_grad_(True) for t in p]
    forward64(q, x, slope).sum().backward()
    ref_g = torch.cat([t.grad.reshape(-1) for t in q])
    got = m.params.grad.cpu().double()
    # a hidden value within rounding of zero may take the other slope: allow one unit's share
    assert (got - ref_g).norm() <= 2e-3 * ref_g.norm()


@pytest.mark.parametrize("power", [-40, -13, 13, 40])
def test_scaled_layers_give_the_same_bits(power):
    """A hidden layer scaled by a power of two and the next one by its inverse is the same network, and every
    scale in the products is a power of two."""
    p = params(5, 28, 3)
    x = (torch.rand((300, 3), generator=torch.Generator().manual_seed(1)) * 2 - 1).to(DEV)
    base = mlp(p, 5, 28, 0.01)(x)
    s = 2.0 ** power
    p[2], p[3], p[4] = p[2] * s, p[3] * s, p[4] / s
    assert torch.equal(mlp(p, 5, 28, 0.01)(x), base)


@pytest.mark.parametrize("scale", [1e-3, 40.0, 4095.0, 4097.0, 3e4])
def test_encoding_ranges_match_fp64(scale):
    p = params(2, 4, 7)
    x = (torch.rand((777, 3), generator=torch.Generator().manual_seed(5)) * 2 - 1) * scale
    # the raw coordinates enter the network too: take their weights out, so that the encoding is what is seen
    p[0][:, :3] = 0.0
    out = mlp(p, 2, 4, 0.0)(x.to(DEV)).detach().cpu().double()
    assert (out - forward64(p, x, 0.0)).abs().max() <= 1e-5


def test_points_do_not_depend_on_their_neighbours():
    p = params(6, 28, 9)
    x = torch.rand((100, 3), generator=torch.Generator().manual_seed(8)) * 2 - 1
    m = mlp(p, 6, 28, 0.01)
    with torch.no_grad():
        base = m(x.to(DEV))
        y = x.clone()
        y[5], y[40] = torch.tensor([5e3, -3e4, 0.1]), float("nan")
        others = [k for k in range(100) if k not in (5, 40)]
        assert torch.equal(m(y.to(DEV))[others], base[others])
        for a, b in ((0, 1), (31, 66), (97, 100)):
            assert torch.equal(m(x[a:b].to(DEV)), base[a:b])
