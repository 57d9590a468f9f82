"""The refinement U-Net's convolutions at the edges of their split: strips of 64 pixels with a remainder, and
row counts per task that do not divide the image.  Weights and activations are FP16 with FP32 sums, so each of
the ten layers adds at most two roundings of 2^-11 of the largest value it carries; a missing or doubled halo
row or column would be of the order of the output itself."""
import pytest
import torch

from snisr import cnn as CN

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


@pytest.mark.parametrize("H,W", [(4, 4), (4, 260), (12, 132), (260, 1284), (1028, 64)])
def test_unet_strip_and_row_remainders(H, W):
    print(f"unet strips {H}x{W}", flush=True)
    torch.manual_seed(H + W)
    net = CN.CNN().eval()
    hip = CN.HipUnet(net, device=DEV)
    g = torch.Generator(device="cpu").manual_seed(W)
    frame = torch.rand(H, W, 3, generator=g).to(DEV)
    inv = (torch.rand(H, W, generator=g) * 0.8 + 0.05).to(DEV)
    bnd = (torch.rand(H, W, generator=g) < 0.1).to(DEV)
    out = hip(frame, inv, bnd)
    torch.cuda.synchronize()
    x = torch.cat([frame.permute(2, 0, 1), inv[None], bnd[None].float()], 0)[None].cpu()
    with torch.no_grad():
        ref = net.cpu().float()(x)[0].permute(1, 2, 0).clamp(0, 1)
    assert float((out.cpu() - ref).abs().max()) <= 20 * 2.0 ** -11 * float(ref.max())
    assert float(ref.std()) > 1e-3
