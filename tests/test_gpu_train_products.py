"""The training MLPs' products hold FP32 operands: all 24 bits of weights, activations and deltas, units of any
scale beside each other, and infinities that stay with the unit they belong to."""
import numpy as np
import pytest
import torch

from snisr import device as D
from snisr import scene as S
from snisr import train as TRN
from snisr import train_ref as TR

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def dims(depth, n_out):
    return [(63 if l == 0 else 64, n_out if l == depth - 1 else 64) for l in range(depth)]


def params(depth, n_out, seed):
    g = torch.Generator().manual_seed(seed)
    out = []
    for i, o in dims(depth, n_out):
        out += [(torch.rand((o, i), generator=g) * 2 - 1) * (6.0 / i) ** 0.5, torch.randn(o, generator=g) * 0.05]
    return out


def points(n, seed):
    return torch.rand((n, 3), generator=torch.Generator().manual_seed(seed)) * 2 - 1


def step(p, x, n_out, slope, g=None):
    """outputs and parameter gradients (per layer weights, biases) of one pass"""
    m = TR.PEMLP(len(p) // 2, n_out, slope, device=DEV)
    with torch.no_grad():
        m.params.copy_(torch.cat([t.reshape(-1) for t in p]))
    out = m(x.to(DEV))
    out.backward(torch.ones_like(out) if g is None else g.to(DEV))
    grads = [t.reshape(q.shape) for t, q in zip(m.params.grad.cpu().split([q.numel() for q in p]), p)]
    return out.detach().cpu(), grads


@pytest.mark.parametrize("depth,n_out", [(2, 4), (6, 28), (8, 4)])
def test_operands_keep_all_bits(depth, n_out):
    """One product per unit (diagonal layers, the encoding of 0 being exactly 0 and 1): every value is the FP32
    product of its two operands, so outputs and bias gradients have one right result."""
    g = torch.Generator().manual_seed(depth)
    w = [torch.rand(64, generator=g) + 0.5 for _ in range(depth)]
    p = []
    for l, (i, o) in enumerate(dims(depth, n_out)):
        W = torch.zeros((o, i))
        if l == 0:
            W[:, 6] = w[0]                              # the input cos(0)
        else:
            W[range(o), range(o)] = w[l][:o]
        p += [W, torch.zeros(o)]
    g_out = torch.randn((1, n_out), generator=g)
    out, grads = step(p, torch.zeros((1, 3)), n_out, 1.0, g_out)
    a = [torch.ones(64), w[0]]                          # inputs of the layers
    for l in range(1, depth):
        a.append(w[l] * a[-1])
    assert torch.equal(out[0], a[-1][:n_out])
    d = g_out[0]
    for l in range(depth - 1, -1, -1):
        assert torch.equal(grads[2 * l + 1], d), l
        if l:
            want = d[:, None].double() * a[l][None, :].double()
            # three 8-bit parts per operand, six of nine products: 2^-25 of the value is left out, FP32 sums add 2^-23
            assert ((grads[2 * l].double() - want).abs() <= 2.0 ** -22 * want.abs()).all(), l
            k = d.numel()
            d = torch.cat([w[l][:k] * d, torch.zeros(64 - k)])


@pytest.mark.parametrize("power", [-45, -30, 30])
@pytest.mark.parametrize("depth,n_out,slope", [(4, 4, 0.0), (6, 28, 0.01)])
def test_scaled_unit_gives_the_same_bits(depth, n_out, slope, power):
    """One hidden unit scaled by a power of two and its outgoing weights by the inverse is the same network."""
    p, x, s, u = params(depth, n_out, 3), points(200, 1), 2.0 ** power, 7
    out, grads = step(p, x, n_out, slope)
    q = [t.clone() for t in p]
    q[2][u] *= s
    q[3][u] *= s
    q[4][:, u] /= s
    out2, grads2 = step(q, x, n_out, slope)
    assert torch.equal(out2, out)
    grads2[2][u] *= s
    grads2[4][:, u] /= s
    # weights only: the four wavefronts of a workgroup add their bias sums with atomics, in no fixed order
    for a, b in zip(grads2[::2], grads[::2]):
        assert torch.equal(a, b)


def test_infinities_stay_in_their_unit():
    p, x = params(3, 28, 5), points(77, 2)
    out, _ = step(p, x, 28, 0.01)
    q = [t.clone() for t in p]
    q[4][3, 11] = float("inf")                          # one weight of output 3
    got, _ = step(q, x, 28, 0.01)
    others = [c for c in range(28) if c != 3]
    assert torch.equal(got[:, others], out[:, others])
    assert not torch.isfinite(got[:, 3]).any()
    p = params(2, 4, 6)
    p[1][9] = float("inf")                              # one infinite activation
    got, _ = step(p, x, 4, 0.0)
    assert torch.equal(got, (p[2][:, 9].sign() * float("inf")).expand(77, 4))


def tile_params(sc):
    """views of the scene's per-tile parameters: (W [T, out, in], b [T, out]) per layer"""
    P, views, at = torch.from_numpy(sc.mlp_params.copy()), [], 0
    for i, o in S.mlp_layer_dims(sc.mlp_in, sc.mlp_width, sc.mlp_layers):
        views.append((P[:, at:at + o * i].view(-1, o, i), P[:, at + o * i:at + o * i + o]))
        at += o * i + o
    return P, views


def render_step(sc, P, o, d, g):
    ds = D.DeviceScene(sc)
    ds.set_params(mlp_params=P.to(DEV))
    out, ws = TRN.train_forward(ds, o, d)
    grads = TRN.train_backward(ds, o, d, g, ws)
    return out, [t.cpu() for t in grads]


@pytest.mark.parametrize("shape", [(16, 32, 3), (16, 64, 3), (32, 128, 4)])
def test_tile_mlp_units_of_any_scale(shape):
    F, width, L = shape
    sc = S.make_scene(11, tile_shape=(2, 1, 1), res=16, occupancy=0.5, feat_dim=F, mlp_width=width, mlp_layers=L,
                      sample_step=1.0 / 48, early_stop=0.0, feat_half=False)
    rng = np.random.default_rng(4)
    t = lambda a: torch.from_numpy(a.astype(np.float32)).to(DEV)  # noqa: E731
    o = rng.uniform([-0.4, -0.4, -0.4], [2.4, 1.4, 1.4], (700, 3))
    d, g = rng.uniform(0.1, 0.9, (700, 3)) * [2, 1, 1] - o, rng.standard_normal((700, 3))
    o, d, g = t(o), t(d), t(g)
    P, _ = tile_params(sc)
    out, grads = render_step(sc, P, o, d, g)
    assert int(out["n_samples"].sum()) > 3000
    s, u = 2.0 ** -30, 5
    Q, v = tile_params(sc)
    v[L - 2][0][:, u] *= s
    v[L - 2][1][:, u] *= s
    v[L - 1][0][:, :, u] /= s
    out2, grads2 = render_step(sc, Q, o, d, g)
    assert torch.equal(out2["rgb"], out["rgb"])
    Q[:] = grads2[2]
    v[L - 2][0][:, u] *= s
    v[L - 2][1][:, u] *= s
    v[L - 1][0][:, :, u] /= s
    for a, b in zip((grads2[0], grads2[1], Q), grads):   # equal but for the order of the atomic sums
        assert (a - b).norm() <= 1e-6 * b.norm()
    # an infinite activation saturates the colours by the sign of its outgoing weights
    Q, v = tile_params(sc)
    v[L - 2][1][:, u] = float("inf")
    v[L - 1][0][:, 0, u], v[L - 1][0][:, 1, u], v[L - 1][0][:, 2, u] = 0.5, -0.5, 0.25
    out3, _ = render_step(sc, Q, o, d, g)
    full = 1.0 - out3["T"]
    assert (out3["rgb"] - torch.stack([full, 0 * full, full], 1)).abs().max() <= 1e-5


# Errors of unbiased sums average out over the 22,000 weights: to 1% of their deviation if independent, a quarter
# leaves room for what they share.  Sums rounded towards one side had a mean of 1.3 to 1.7 deviations here.
@pytest.mark.parametrize("depth,n_out", [(6, 28), (8, 4)])
def test_weight_gradients_are_not_biased(depth, n_out):
    n = 64 * 8281
    p, x = params(depth, n_out, 1), points(n, 1)
    g = torch.randn((n, n_out), generator=torch.Generator().manual_seed(2))
    _, grads = step(p, x, n_out, 1.0, g)
    q = [t.double().to(DEV).requires_grad_(True) for t in p]
    x = x.double().to(DEV)
    h = torch.cat([x] + [f((2.0 ** k) * x) for k in range(10) for f in (torch.sin, torch.cos)], 1)
    for l in range(depth):
        h = h @ q[2 * l].T + q[2 * l + 1]
    h.backward(g.double().to(DEV))
    err = torch.cat([(a.double() - t.grad.cpu()).reshape(-1) for a, t in zip(grads[::2], q[::2])])
    assert abs(err.mean()) <= 0.25 * err.std()
