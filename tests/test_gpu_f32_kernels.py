"""The 32-bit path's products on the float matrix cores against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def ops():
    from reinfer_amd import kernels
    return kernels.current()


# rows on both sides of the two kernels' edges (16, 32, 64, 128), features off every tile (of 64 and, with many, of 128), k with a part piece of 32, a last
# range shorter than the others, and rows that are no 16-byte pieces (the plain kernel's)
@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 64, 65, 129, 300])
@pytest.mark.parametrize("N,K", [(16, 32), (7, 4), (100, 68), (333, 2052), (1030, 1120), (40, 6144), (24, 70), (4100, 2052), (8193, 516)])
@pytest.mark.parametrize("bias", [False, True])
def test_product_of_float_matrices(M, N, K, bias):
    g = torch.Generator(device=DEV).manual_seed(M * N + K)
    wide = torch.randn(M, K + 4, generator=g, device=DEV)
    x = wide[:, :K]                                        # rows longer than the product's
    w = torch.randn(N, K, generator=g, device=DEV)
    b = torch.randn(N, generator=g, device=DEV) if bias else None
    buf = torch.full((M, N + 3), 7.0, device=DEV)
    out = buf[:, :N]
    ops().linear(x, w, out, b)
    want = x.double() @ w.double().t() + (b.double() if bias else 0.0)
    # a sum of K float products in any order: at most (K + 2) roundings of half an ulp of the sum of magnitudes
    bound = (K + 2) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + (b.double().abs() if bias else 0.0))
    assert ((out.double() - want).abs() <= bound).all()
    assert (buf[:, N:] == 7.0).all()


def test_product_of_float_matrices_is_exact_where_floats_are():
    """Small whole numbers: every product and sum is exact, so any order gives the same bits, and a value that a lower
    precision would round away stays."""
    g = torch.Generator(device=DEV).manual_seed(3)
    for M in (5, 40, 200):
        x = torch.randint(-512, 513, (M, 256), generator=g, device=DEV).float()
        w = torch.randint(-64, 65, (96, 256), generator=g, device=DEV).float()
        out = torch.empty(M, 96, device=DEV)
        ops().linear(x, w, out)
        assert torch.equal(out.double(), x.double() @ w.double().t())
