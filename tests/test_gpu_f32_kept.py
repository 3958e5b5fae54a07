"""What the 32-bit products keep of floats: numbers down to the smallest and up to the largest, mantissas that the six terms serve worst,
errors without a mean, many sums that are not finite; and a row's bits beside any others."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
U = 2.0 ** -24
ROWS = [1, 8, 9, 16, 17, 32, 33, 64, 65, 160, 300, 1100]          # every form of both kernels, cut and whole


def product(x, w, bias=None):
    from reinfer_amd import kernels
    out = torch.empty(x.shape[0], w.shape[0], device=DEV)
    kernels.current().linear(x, w, out, bias)
    return out


def blocks(K):
    """How many blocks K is summed in, and k of one."""
    n = min(8, max(1, K // 512))
    k = -(-(-(-K // n)) // 64) * 64
    return -(-K // k), k


def spread(K):
    """Of sums of K products of independent signs, the error's norm over the result's: a block's large terms are rounded into their sum once
    for every eight k, the two sums and the blocks' once each; a rounding is at most U of what it rounds and spread evenly (3 ** -0.5 of that
    in the mean square). All six terms rounded into one sum: sqrt(6) of the first part."""
    n, k = blocks(K)
    return U * ((k / 16 + n / 2 + 1) / 3) ** 0.5


def most(K):
    """The same, were all errors of one sign: U of a product is left out as well."""
    n, k = blocks(K)
    return U * (1 + 2.0 ** -8 + k / 8 + n + 1)


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("K", [512, 1092, 2560, 9728])
def test_errors_are_small_and_have_no_mean(M, K):
    g = torch.Generator(device=DEV).manual_seed(M + K)
    x, w = torch.randn(M, K, generator=g, device=DEV), torch.randn(520, K, generator=g, device=DEV) * 0.02
    want = x.double() @ w.double().t()
    off = product(x, w).double() - want
    assert off.norm() / want.norm() < spread(K)
    assert off.mean().abs() / want.std() < 16 * spread(K) / want.numel() ** 0.5


@pytest.mark.parametrize("M", ROWS)
@pytest.mark.parametrize("e", [-90, -109, -116, -124, -127, -133, -140])
def test_small_numbers_are_whole(M, e):
    """Rows of 2^e, down to where floats are subnormal, by large weights; and the other way round."""
    g = torch.Generator(device=DEV).manual_seed(M - e)
    K = 1028
    small, large = torch.randn(M, K, generator=g, device=DEV) * 2.0 ** e, torch.randn(72, K, generator=g, device=DEV) * 2.0 ** 40
    for x, w in ((small, large), (torch.randn(M, K, generator=g, device=DEV) * 2.0 ** 40, torch.randn(72, K, generator=g, device=DEV) * 2.0 ** e)):
        want = x.double() @ w.double().t()
        assert (product(x, w).double() - want).norm() / want.norm() < spread(K)


@pytest.mark.parametrize("M", [1, 9, 32, 64, 160, 300])
def test_worst_mantissas(M):
    """1 + 2^-8 - 2^-17 is 1, 2^-8 and -2^-17: what is left out of its square is 0.99 of U, and all of one sign."""
    a = 1 + 2.0 ** -8 - 2.0 ** -17
    g = torch.Generator(device=DEV).manual_seed(M)
    for K in (512, 4096):
        x, w = torch.full((M, K), a, device=DEV), torch.full((200, K), a, device=DEV)
        for sign in (torch.ones(200, K, device=DEV), torch.randint(0, 2, (200, K), generator=g, device=DEV) * 2.0 - 1.0):
            want = x.double() @ (w * sign).double().t()
            assert ((product(x, w * sign).double() - want).abs() <= most(K) * K * a * a).all()
    # a single product: what is left out of it and one rounding, where a float product has the rounding
    x, w = torch.zeros(M, 512, device=DEV), torch.zeros(200, 512, device=DEV)
    x[:, 37], w[:, 37] = torch.rand(M, generator=g, device=DEV) + 1, torch.rand(200, generator=g, device=DEV) + 1
    x[0, 37] = w[0, 37] = a
    want = x.double() @ w.double().t()
    assert ((product(x, w).double() - want).abs() <= (2 + 2.0 ** -6) * U * want).all()


@pytest.mark.parametrize("M", ROWS)
def test_many_that_are_not_finite(M):
    """Whole rows, and all of them, that hold an infinity or a NaN; sums past 2^80, which are worked out from the floats."""
    g = torch.Generator(device=DEV).manual_seed(M)
    K, N = 1092, 140
    x, w = torch.randn(M, K, generator=g, device=DEV), torch.randn(N, K, generator=g, device=DEV)
    for rows in (slice(0, M, 3), slice(0, M)):
        for value in (float("inf"), float("nan")):
            y = x.clone()
            y[rows, 700] = value
            want = (y.double() @ w.double().t()).float()
            got = product(y, w)
            assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got[want.isinf()], want[want.isinf()])
            keep = want.isfinite()
            assert torch.equal(got[keep], product(x, w)[keep])
    y = x.clone()
    y[::2] *= 2.0 ** 90
    want = y.double() @ w.double().t()
    got = product(y, w)
    assert ((got.double() - want).abs() <= (K + 8) * U * (y.double().abs() @ w.double().abs().t())).all()


@pytest.mark.parametrize("N,K", [(2560, 1092), (200, 4096), (6144, 2560)])
def test_a_rows_bits_beside_any_others(N, K):
    g = torch.Generator(device=DEV).manual_seed(N)
    x, w, b = torch.randn(1100, K, generator=g, device=DEV), torch.randn(N, K, generator=g, device=DEV), torch.randn(N, generator=g, device=DEV)
    x[5] *= 2.0 ** 90                      # past the range of the parts' sums
    x[6] *= 2.0 ** -130
    x[7, 3] = 3.4e38
    whole = product(x, w, b)
    for M in ROWS[:-1]:
        part = product(x[:M], w, b)
        assert torch.equal(part.view(torch.int32), whole[:M].view(torch.int32)), M
    for m in (5, 6, 7, 1099):
        assert torch.equal(product(x[m:m + 1], w, b).view(torch.int32), whole[m:m + 1].view(torch.int32)), m


@pytest.mark.parametrize("M,N,K,rows", [(8, 2560, 9728, 1), (4, 6144, 2560, 4), (300, 6144, 2560, 1), (300, 2560, 2560, 300)])
def test_what_is_not_finite_costs_a_few_products(M, N, K, rows):
    """What is worked out again is shared out over whole waves: some ten times the product at most, all of it NaN (3 to 6 measured; a lane a
    sum took 20 to 50)."""
    x, w = torch.randn(M, K, device=DEV), torch.randn(N, K, device=DEV)

    def time(x):
        out, best = torch.empty(M, N, device=DEV), float("inf")
        from reinfer_amd import kernels
        for _ in range(8):
            first, last = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            first.record()
            for _ in range(4):
                kernels.current().linear(x, w, out, None)
            last.record()
            torch.cuda.synchronize()
            best = min(best, first.elapsed_time(last))
        return best
    plain = time(x)
    x[:rows, 5] = float("nan")
    assert time(x) < 10 * plain
