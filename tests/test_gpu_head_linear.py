"""Products head by head in bfloat16 with rows that four-column accesses can take, against float64."""
import pytest
import torch

from reinfer_amd import kernels

pytestmark = pytest.mark.gpu
DEV = "cuda"


# tokens on both sides of 16 and 64; K with a half step of 64, a part of a step of 32 and one step alone; columns that end
# inside a wave's 16 and inside a workgroup's 64
@pytest.mark.parametrize("T", [1, 16, 17, 64, 65, 131])
@pytest.mark.parametrize("H,K,N", [(2, 128, 192), (3, 192, 128), (2, 40, 20), (1, 8, 4), (5, 96, 68)])
@pytest.mark.parametrize("gated", ["no", "columns", "heads"])
def test_head_products_in_whole_pieces(T, H, K, N, gated):
    g = torch.Generator(device=DEV).manual_seed(T * K + N)
    x = torch.randn(T, H * K + 8, generator=g, device=DEV).to(torch.bfloat16)[:, 8:]
    w = (torch.randn(H, N, K, generator=g, device=DEV) / K ** 0.5).to(torch.bfloat16)
    gate = torch.randn(T, H * N if gated == "columns" else H + 3, generator=g, device=DEV).to(torch.bfloat16)
    out = torch.full((T, H * (N + 4)), float("nan"), device=DEV, dtype=torch.bfloat16)
    more = {"gate": gate[:, :H] if gated == "heads" else gate, "gate_per_head": gated == "heads"} if gated != "no" else {}
    kernels.current().head_linear(x, K, w, out, N + 4, **more)
    xs, wd = x.double().view(T, H, K), w.double()
    want = (xs.transpose(0, 1) @ wd.transpose(1, 2)).transpose(0, 1)
    mags = (xs.abs().transpose(0, 1) @ wd.abs().transpose(1, 2)).transpose(0, 1)
    if gated != "no":
        want = want * torch.sigmoid(gate.double()[:, :H, None] if gated == "heads" else gate.double().view(T, H, N))
    got = out.view(T, H, N + 4)
    # K + 4 float roundings of the sum of magnitudes, then one to bfloat16
    assert ((got[..., :N].double() - want).abs() <= mags * (K + 4) * 2.0 ** -24 + want.abs() * 2.0 ** -8).all()
    assert torch.isnan(got[..., N:]).all()
