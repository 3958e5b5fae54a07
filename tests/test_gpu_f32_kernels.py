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


# off every tile and block of K; with many rows uncut, with few cut into ranges of blocks
@pytest.mark.parametrize("N,K,most_x,most_w", [(96, 516, 4095, 7), (1030, 1540, 4095, 2), (333, 6148, 2701, 1), (40, 512, 4095, 7),
                                               (19456, 2560, 4095, 1)])
def test_float_matrix_cores_are_exact_where_floats_are(N, K, most_x, most_w):
    """Whole numbers of up to 12 bits whose sums stay below 2^24 in any order: every bit counts, whichever kernel runs."""
    from reinfer_amd.kernels import library
    assert K * most_x * most_w < 2 ** 24
    g = torch.Generator(device=DEV).manual_seed(K)
    w = torch.randint(-most_w, most_w + 1, (N, K), generator=g, device=DEV).float()
    for M in (1, 16, 17, 32, 33, 64, 65, 200, 1100):
        x = torch.randint(-most_x, most_x + 1, (M, K), generator=g, device=DEV).float()
        assert library.load().ra_gemm_f32_supports(x.data_ptr(), w.data_ptr(), K, K) == 1
        out = torch.empty(M, N, device=DEV)
        ops().linear(x, w, out)
        assert torch.equal(out.double(), x.double() @ w.double().t()), M


# one to eight blocks of K, the last of them short; features off the tiles
@pytest.mark.parametrize("N,K", [(40, 512), (8193, 516), (1030, 1120), (333, 2052), (6144, 2560), (2560, 4096), (100, 6144), (2560, 9728)])
@pytest.mark.parametrize("bias", [False, True])
def test_a_row_has_the_same_bits_whatever_stands_beside_it(N, K, bias):
    g = torch.Generator(device=DEV).manual_seed(N + K)
    x = torch.randn(1300, K, generator=g, device=DEV)
    w = torch.randn(N, K, generator=g, device=DEV)
    b = torch.randn(N, generator=g, device=DEV) if bias else None
    want = torch.empty(1300, N, device=DEV)
    ops().linear(x, w, want, b)
    for M in (1, 5, 16, 17, 31, 32, 33, 64, 65, 129, 300, 700):
        out = torch.empty(M, N, device=DEV)
        ops().linear(x[1300 - M:], w, out, b)
        assert torch.equal(out, want[1300 - M:]), M
