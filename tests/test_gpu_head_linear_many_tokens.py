"""Products head by head with many tokens (four column tiles a wave) and just below that, against float64."""
import pytest
import torch

from reinfer_amd import kernels

pytestmark = pytest.mark.gpu
DEV = "cuda"


# waves for every SIMD just reached and just not (32 tokens by 64 columns by heads); token tiles that end inside a wave, a workgroup;
# K in one step, steps with 8 left, several; columns that are no whole tiles of 64
@pytest.mark.parametrize("T,H,N,K", [(993, 16, 128, 192), (992, 16, 128, 192), (2049, 16, 64, 8), (1300, 8, 192, 72),
                                     (4095, 8, 64, 128), (1000, 16, 132, 64)])
@pytest.mark.parametrize("gate", [None, "column", "head"])
def test_many_tokens(T, H, N, K, gate):
    g = torch.Generator(device=DEV).manual_seed(T + N)
    x = torch.randn(T, H * (K + 8), device=DEV, generator=g).bfloat16()
    w = (torch.randn(H, N, K, device=DEV, generator=g) / K ** 0.5).bfloat16()
    out = torch.full((T + 1, H * (N + 4)), float("nan"), device=DEV, dtype=torch.bfloat16)
    gates = None if gate is None else torch.randn(T, H * N if gate == "column" else H, device=DEV, generator=g).bfloat16()
    kernels.current().head_linear(x, K + 8, w, out[:T], N + 4, gates, gate == "head")
    xd = x.double().view(T, H, K + 8)[:, :, :K].transpose(0, 1).contiguous()
    wd = w.double().transpose(1, 2).contiguous()
    want, size = torch.bmm(xd, wd).transpose(0, 1), torch.bmm(xd.abs(), wd.abs()).transpose(0, 1)
    if gate is not None:
        s = torch.sigmoid(gates.double()).view(T, H, -1)
        want, size = want * s, size * s
    got = out[:T].view(T, H, N + 4)
    # K float roundings of at most 2^-24 of the magnitudes, the hardware's exponential, and the result's own rounding
    assert ((got[:, :, :N].double() - want).abs() <= size * (K * 2.0 ** -24 + 2.0 ** -20) + want.abs() * 2.0 ** -8).all()
    assert torch.isnan(got[:, :, N:]).all() and torch.isnan(out[T]).all()
