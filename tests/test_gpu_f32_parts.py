"""The 32-bit products' floats in three parts, where a part can go wrong: infinities, NaN and the largest floats, one row among
others; numbers over the whole range of exponents; and the error against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ROWS = [1, 8, 9, 16, 17, 32, 33, 64, 65, 160, 250, 1100]          # every form of both kernels, cut and whole


def product(x, w, bias=None):
    from reinfer_amd import kernels
    out = torch.empty(x.shape[0], w.shape[0], device=DEV)
    kernels.current().linear(x, w, out, bias)
    return out


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("N,K", [(136, 1092), (2560, 4096)])
def test_what_is_not_finite_comes_out_as_of_floats(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M + K)
    x, w = torch.randn(M, K, generator=g, device=DEV), torch.randn(N, K, generator=g, device=DEV)
    b = torch.randn(N, generator=g, device=DEV)
    plain = product(x, w, b)
    m = M // 2
    w[7, :8] = torch.tensor([1.0, -2.0, 0.5, 4.0, 0.0, 1.0, -1.0, 2.0], device=DEV)      # one part, and a zero
    for value in (float("inf"), float("-inf"), float("nan"), 3.4e38, -3.4028234e38):
        y = x.clone()
        y[m, 3] = value
        got, want = product(y, w, b), (y[m:m + 1].double() @ w.double().t() + b.double())[0].float()
        if abs(value) < float("inf"):           # what is within a rounding of the largest float is neither's to say
            near = (want.abs() > 3.3e38) & (want.abs() < 3.5e38)
            finite = want.isfinite() & ~near
            assert ((got[m] - want).abs()[finite] <= 2.0 ** -20 * 3.4e38).all()
            assert torch.equal(got[m][~want.isfinite() & ~near], want[~want.isfinite() & ~near])
        else:
            assert torch.equal(got[m].isnan(), want.isnan())
            assert torch.equal(got[m][~want.isnan()], want[~want.isnan()])
        keep = torch.arange(M, device=DEV) != m
        cols = torch.arange(N, device=DEV) != 7
        assert torch.equal(got[keep][:, cols], plain[keep][:, cols])      # the rows beside it keep their bits


@pytest.mark.parametrize("M", ROWS)
def test_exponents_of_all_sizes(M):
    """Rows and weights of 2^-60 .. 2^60: every product is a float's, and each is off by no more than its own roundings. What the six
    terms leave out is some 2^-24 of a product, the sum's roundings are four for every 32 k and two for each of its blocks; six and one are
    granted, twice over."""
    g = torch.Generator(device=DEV).manual_seed(M)
    K, N = 2052, 100

    def spread(*shape):
        e = torch.randint(-60, 61, shape, generator=g, device=DEV).float()
        return torch.randn(*shape, generator=g, device=DEV) * torch.exp2(e)
    x, w = spread(M, K), spread(N, K)
    want = x.double() @ w.double().t()
    bound = (K * 6 / 32 + 8 + 2) * 2.0 ** -24 * 2 * (x.double().abs() @ w.double().abs().t())
    assert ((product(x, w).double() - want).abs() <= bound).all()


# the least errors that full float products with float sums of these lengths showed on the same numbers were 4.0e-7, 4.0e-7 and 6.2e-7
@pytest.mark.parametrize("K,most", [(2560, 3.9e-7), (4096, 3.9e-7), (9728, 6.1e-7)])
def test_error_against_64_bits(K, most):
    g = torch.Generator(device=DEV).manual_seed(K)
    w = torch.randn(512, K, generator=g, device=DEV) * 0.02
    for M in (4, 32, 300, 1100):
        x = torch.randn(M, K, generator=g, device=DEV)
        want = x.double() @ w.double().t()
        assert (product(x, w).double() - want).norm() / want.norm() < most
