"""The tiled bfloat16 product of 65 to 512 rows against float64, at the edges of its tiles, K ranges and dispatch."""
import math

import pytest
import torch

from reinfer_amd import kernels

pytestmark = pytest.mark.gpu
DEV = "cuda"


def ops():
    return kernels.current()


def operands(M, N, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K, device=DEV, generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV, generator=g) / math.sqrt(K)).to(torch.bfloat16)
    return x, w, g


def bound(x, w, K):
    """Float sums of K exact products in any order: K roundings of at most 2^-24 of the sum of magnitudes, which the
    matrix cores' own order halves many times over; a twentieth of that worst case still catches a lost or doubled k."""
    return (x.double().abs() @ w.double().abs().T) * (K * 2.0 ** -24 / 20) + 1e-6


# row tiles of 128 at, below and above their edges; feature tiles with 1, 4 and 127 left; K with pieces left of a step of 64
# and of a range; two ranges and many
SIZES = [(65, 4096, 4096), (97, 6144, 4096), (128, 4097, 1032), (129, 2564, 4096), (192, 1151, 6152), (256, 4096, 12288),
         (255, 8128, 1536), (257, 4224, 8192), (512, 2560, 9736), (511, 2049, 8200), (65, 7936, 1024)]


@pytest.mark.parametrize("M,N,K", SIZES)
def test_tiled_product_with_each_epilogue(M, N, K):
    lib = kernels.library.load()
    assert lib.ra_gemm_tile_takes(0, M, N, K) == 1
    x, w, g = operands(M, N, K, M + N)
    ref, err = x.double() @ w.double().T, bound(x, w, K)
    bias = torch.randn(N, device=DEV, generator=g).to(torch.bfloat16)
    out = torch.full((M, N), float("nan"), device=DEV)
    ops().linear(x, w, out)
    assert ((out.double() - ref).abs() <= err).all()
    ops().linear(x, w, out, bias)
    biased = ref + bias.double()
    assert ((out.double() - biased).abs() <= err + biased.abs() * 2 ** -23).all()
    half = torch.full((M, N + 4), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops().linear(x, w, half[:, :N], bias)               # rows that are not next to one another
    assert ((half[:, :N].double() - biased).abs() <= err + biased.abs() * 2 ** -8).all()
    assert torch.isnan(half[:, N:]).all()
    for alpha in (1.0, 0.25):
        stream = torch.randn(M, N, device=DEV, generator=g) * 8
        want = stream.double() + alpha * ref
        ops().linear_skinny(x, w, stream, accumulate=True, alpha=alpha)
        assert ((stream.double() - want).abs() <= err + want.abs() * 2 ** -23).all()
    parts = ops().linear_ranges(x, w)
    assert parts.shape[0] == lib.ra_gemm_wide_ranges(M, N, K) >= 2
    assert ((parts.double().sum(0) - ref).abs() <= err).all()


@pytest.mark.parametrize("M,I,K", [(65, 9728, 2560), (97, 12288, 4096), (128, 16384, 1024), (128, 8200, 1032)])
def test_tiled_gated_product(M, I, K):
    assert kernels.library.load().ra_gemm_tile_takes(1, M, 2 * I, K) == 1
    x, w, _ = operands(M, 2 * I, K, M + I)
    out = torch.full((M, I), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops().gated_linear(x, w, out)
    prod, err = x.double() @ w.double().T, bound(x, w, K)
    rows = torch.arange(2 * I, device=DEV).view(-1, 2, 8)
    gate, up = prod[:, rows[:, 0].reshape(-1)], prod[:, rows[:, 1].reshape(-1)]
    eg, eu = err[:, rows[:, 0].reshape(-1)], err[:, rows[:, 1].reshape(-1)]
    want = gate * torch.sigmoid(gate) * up              # silu's slope is at most 1.1
    assert ((out.double() - want).abs() <= 1.1 * eg * (up.abs() + eu) + gate.abs() * eu + want.abs() * (2 ** -8 + 2 ** -20)).all()


def test_tiled_product_takes_only_what_it_can_read():
    """Sizes past its rule, rows of no whole 16-byte pieces and unaligned pointers stay with the library's product."""
    lib = kernels.library.load()
    for epilogue, M, N, K in [(0, 64, 4096, 4096), (0, 513, 4096, 12288), (0, 257, 4096, 4096), (0, 97, 22528, 4096),
                              (0, 384, 4096, 12288), (0, 97, 512, 1024), (1, 129, 24576, 4096), (1, 97, 4096, 4096)]:
        assert lib.ra_gemm_tile_takes(epilogue, M, N, K) == 0
    M, N, K = 97, 4096, 4096
    x, w, g = operands(M, N, K + 8, 3)
    odd = torch.empty(M, K + 12, device=DEV, dtype=torch.bfloat16)[:, 1:K + 1]
    odd.copy_(x[:, :K])
    rows = torch.randn(1, K, device=DEV, generator=g).to(torch.bfloat16).expand(M, K)
    w = w[:, :K].contiguous()
    for a in (odd, rows):
        assert not ops()._tile_takes(0, a, w, torch.empty(M, N, device=DEV, dtype=torch.bfloat16))
        out = torch.full((M, N), float("nan"), device=DEV, dtype=torch.bfloat16)
        ops().linear(a, w, out)
        want = a.double() @ w.double().T
        assert ((out.double() - want).abs() <= bound(a, w, K) + want.abs() * 2 ** -8).all()


@pytest.mark.parametrize("dtype,M,K", [(torch.bfloat16, M, 4096) for M in (8, 97, 200, 600)] + [(torch.float32, M, 512) for M in (8, 97)])
def test_a_bias_that_is_a_column_of_a_matrix(dtype, M, K):
    N = 4096
    x, w, g = operands(M, N, K, M)
    x, w = x.to(dtype), w.to(dtype)
    biases = torch.randn(N, 3, device=DEV, generator=g).to(dtype)
    out, want = torch.empty(M, N, device=DEV, dtype=dtype), torch.empty(M, N, device=DEV, dtype=dtype)
    ops().linear(x, w, out, biases[:, 1])
    ops().linear(x, w, want, biases[:, 1].clone())
    assert torch.equal(out, want)


@pytest.mark.parametrize("M,N,K", SIZES)
def test_tiled_product_where_the_library_is_asked_first(M, N, K):
    """The kernel itself at every size it takes, also where ``linear`` prefers the library's product."""
    x, w, g = operands(M, N, K, M * 3 + N)
    ref, err = x.double() @ w.double().T, bound(x, w, K)
    bias = torch.randn(N, device=DEV, generator=g).to(torch.bfloat16)
    biased = ref + bias.double()
    for kind, ulp in ((torch.float32, 2.0 ** -23), (torch.bfloat16, 2.0 ** -8)):
        buf = torch.full((M, N + 8), float("nan"), device=DEV, dtype=kind)
        ops()._few_rows("linear output", x, w, bias, buf[:, :N], 0, M, N, K, True)
        assert ((buf[:, :N].double() - biased).abs() <= err + biased.abs() * ulp).all()
        assert torch.isnan(buf[:, N:]).all()
    stream = torch.randn(M, N, device=DEV, generator=g) * 8
    want = stream.double() + ref
    ops()._few_rows("linear output", x, w, None, stream, 2, M, N, K, True)
    assert ((stream.double() - want).abs() <= err + want.abs() * 2 ** -23).all()


def test_small_cut_products_stay_with_the_library():
    def takes(epilogue, M, N, K):
        x, w = torch.empty(M, K, device=DEV, dtype=torch.bfloat16), torch.empty(N, K, device=DEV, dtype=torch.bfloat16)
        return ops()._tile_takes(epilogue, x, w, torch.empty(M, N, device=DEV, dtype=torch.float32 if epilogue == 2 else torch.bfloat16))
    for M in (65, 128, 256):
        assert not any(takes(0, M, N, K) for N, K in ((8192, 2048), (6144, 2560), (4096, 4096)))
        assert takes(0, M, 6144, 4096) and takes(0, M, 4096, 6144)
    assert takes(2, 97, 2560, 4096) and takes(2, 160, 2560, 4096) and takes(2, 160, 2560, 9728) and takes(1, 97, 24576, 4096)


def test_rows_too_far_apart_to_address_stay_with_the_library():
    """512 rows of 2^21 elements are more than a descriptor covers: such calls went to the library's product, and still do."""
    M, N, K = 512, 4096, 12288
    w = torch.empty(N, K, device=DEV, dtype=torch.bfloat16)
    for stride, taken in ((K, True), (2 ** 20 - 8, True), (2 ** 20, False), (2 ** 21 - 8, False)):
        x = torch.empty((M - 1) * stride + K, device=DEV, dtype=torch.bfloat16).as_strided((M, K), (stride, 1))
        assert ops()._tile_takes(2, x, w, torch.empty(M, N, device=DEV)) == taken
        assert taken or ops().linear_ranges(x, w) is None


# a width of tile each (64, 80, 96, 112, 128, 160 features; fewer tiles than CUs, one more than they are, and several rounds), N and K at
# and off whole tiles, stages and pieces of four, rows on both sides of a tile of 16 and of the 32 and 64 that the kernel is built for
@pytest.mark.parametrize("M", [16, 17, 32, 33, 49, 64])
@pytest.mark.parametrize("N,K", [(19456, 264), (24576, 320), (51200, 128), (151936, 72), (40016, 640), (32896, 8), (6144, 2560), (2560, 4104)])
def test_few_rows_in_tiles_of_every_width(M, N, K):
    """Plain results in both types, with and without a bias and at a stride that is in no whole pieces; added; gated."""
    x, w, g = operands(M, N, K, M + N + K)
    ref, err = x.double() @ w.double().T, bound(x, w, K)
    bias = torch.randn(N, device=DEV, generator=g).to(torch.bfloat16)
    for kind, ulp in ((torch.float32, 2.0 ** -23), (torch.bfloat16, 2.0 ** -8)):
        for wide, b in ((N + 8, None), (N + 8, bias), (N + 3, None)):
            buf = torch.full((M, wide), float("nan"), device=DEV, dtype=kind)
            ops().linear_skinny(x, w, buf[:, :N], b, wide=True)
            want = ref if b is None else ref + b.double()
            assert ((buf[:, :N].double() - want).abs() <= err + want.abs() * ulp).all()
            assert torch.isnan(buf[:, N:]).all()
    stream = torch.randn(M, N, device=DEV, generator=g)
    want = stream.double() + ref
    ops().linear_skinny(x, w, stream, accumulate=True, wide=True)
    assert ((stream.double() - want).abs() <= err + want.abs() * 2 ** -23).all()
    out = torch.full((M, N // 2), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops().gated_linear(x, w, out, wide=True)
    rows = torch.arange(N, device=DEV).view(-1, 2, 8)
    gate, up = ref[:, rows[:, 0].reshape(-1)], ref[:, rows[:, 1].reshape(-1)]
    eg, eu = err[:, rows[:, 0].reshape(-1)], err[:, rows[:, 1].reshape(-1)]
    want = gate * torch.sigmoid(gate) * up
    assert ((out.double() - want).abs() <= 1.1 * eg * (up.abs() + eu) + gate.abs() * eu + want.abs() * (2 ** -8 + 2 ** -20)).all()


@pytest.mark.parametrize("M", [17, 48, 64])
@pytest.mark.parametrize("parts", [1, 4, 5, 8, 9, 160, 257])
def test_a_carried_norm_of_any_number_of_parts(M, parts):
    N, K, eps = 24576, 192, 1e-6
    x, w, g = operands(M, N, K, parts)
    ss = torch.rand(parts, M, device=DEV, generator=g) + 0.1
    factor = torch.rsqrt(ss.double().sum(0) / K + eps)[:, None]
    out = torch.full((M, N), float("nan"), device=DEV)
    ops().linear_skinny(x, w, out, row_sums=(ss, eps, K))
    want = x.double() @ w.double().T * factor
    # the sums of the parts and the factor: parts + 4 roundings at most
    assert ((out.double() - want).abs() <= bound(x, w, K) * factor + want.abs() * (parts + 4) * 2 ** -24).all()


def test_a_gate_of_what_is_not_finite():
    """silu of infinities and of what overflows: as the float formula has them."""
    M, I, K = 17, 12288, 64
    x, w = torch.zeros(M, K, device=DEV, dtype=torch.bfloat16), torch.zeros(2 * I, K, device=DEV, dtype=torch.bfloat16)
    x[:, 0] = 1
    gate = torch.tensor([0.0, 1e30, -1e30, 88.0, -88.0, 130.0, -130.0, float("inf"), float("-inf"), float("nan")], device=DEV).to(torch.bfloat16)
    rows = torch.arange(2 * I, device=DEV).view(-1, 2, 8)
    w[rows[:, 0].reshape(-1)[:len(gate)], 0] = gate
    w[rows[:, 1].reshape(-1), 0] = 1
    out = torch.empty(M, I, device=DEV, dtype=torch.bfloat16)
    ops().gated_linear(x, w, out, wide=True)
    v = gate.float()
    want = torch.where(v <= -88, v * 0, v * torch.sigmoid(v))
    want[8] = float("nan")                  # minus infinity over infinity
    got = out[0, :len(gate)].float()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.allclose(got.nan_to_num(0.0, 1e38, -1e38), want.nan_to_num(0.0, 1e38, -1e38), rtol=2 ** -8, atol=1e-30)


# 65 to 128 rows, the first and the last N of a width of tile (80, 96, 112, 128 features)
@pytest.mark.parametrize("M", [65, 113, 128])
@pytest.mark.parametrize("I,K", [(8200, 1032), (10240, 1024), (10248, 1032), (12288, 1096), (12296, 1032), (14336, 1536), (14344, 1032)])
def test_gated_in_tiles_of_every_width(M, I, K):
    test_tiled_gated_product(M, I, K)


# planes in tiles of 64, 80, 96, 112 and 128 features above 64 rows, and of 80, 96, 112, 128 and 160 below; N off a whole tile, ranges
# that end inside a stage
@pytest.mark.parametrize("M,N,K", [(M, N, K) for M in (65, 97, 128) for N, K in ((4096, 4104), (10236, 2568), (6144, 4104), (7168, 4104),
                                                                               (2564, 12296), (7164, 2056))]
                         + [(M, N, K) for M in (17, 33, 64) for N, K in ((2560, 4104), (4604, 2568), (7164, 2568), (6656, 4096), (10236, 4104),
                                                                         (9216, 4096))])
def test_planes_in_tiles_of_every_width(M, N, K):
    lib = kernels.library.load()
    x, w, g = operands(M, N, K, M * 5 + N)
    ref, err = x.double() @ w.double().T, bound(x, w, K)
    S = int(lib.ra_gemm_wide_ranges(M, N, K))
    parts = torch.full((S, M, N), float("nan"), device=DEV)
    for keep in (0, 1):
        if M > 64 and not lib.ra_gemm_tile_takes(0, M, N, K):
            break
        kernels.library.call("ra_gemm_wide_partial", x.data_ptr(), w.data_ptr(), parts.data_ptr(), parts.numel(), M, N, K, K, keep,
                             torch.cuda.current_stream().cuda_stream)
        assert ((parts.double().sum(0) - ref).abs() <= err).all()
        parts.fill_(float("nan"))
    stream = torch.randn(M, N, device=DEV, generator=g)
    want = stream.double() + ref
    ops()._few_rows("linear output", x, w, None, stream, 2, M, N, K, True)
    assert ((stream.double() - want).abs() <= err + want.abs() * 2 ** -23).all()


@pytest.mark.parametrize("N", [16, 33000])          # one tile in ranges of K; tiles of 160 features where K allows them
def test_rows_too_long_for_the_widest_tile(N):
    """160 rows of weights span more than a descriptor covers, 128 do not: a narrower tile takes the product."""
    M, K = 17, 6710912 if N == 16 else 128
    x, w, _ = operands(M, N, K, 5)
    out = torch.full((M, N), float("nan"), device=DEV)
    ops().linear_skinny(x, w, out, wide=True)
    for n in range(0, N, 4096):
        part = slice(n, n + 4096)
        want = sum(x[:, k:k + (1 << 20)].double() @ w[part, k:k + (1 << 20)].double().T for k in range(0, K, 1 << 20))
        # sums of deviation 1, rounded K times at most by up to 2^-25 in either direction: eight deviations of their sum, a fifth of
        # what a lost stage of 64 k would show
        assert ((out[:, part].double() - want).abs() <= 8 * math.sqrt(K) * 2 ** -25 * (1 + want.abs())).all()


@pytest.mark.parametrize("M", [17, 64, 128])
@pytest.mark.parametrize("N,K", [(8192, 4096), (4096, 4104), (7168, 4104), (6144, 4096)])
def test_four_ranges_each_in_its_plane(M, N, K):
    """Four ranges, which panels of weights start one on from one another, land where the adding kernels look for them."""
    x, w, _ = operands(M, N, K, M + N)
    S = int(kernels.library.load().ra_gemm_wide_ranges(M, N, K))
    assert S == 4
    parts = torch.full((S, M, N), float("nan"), device=DEV)
    kernels.library.call("ra_gemm_wide_partial", x.data_ptr(), w.data_ptr(), parts.data_ptr(), parts.numel(), M, N, K, K, 0,
                         torch.cuda.current_stream().cuda_stream)
    each = (-(-K // S) + 63) // 64 * 64
    for z in range(S):
        xs, ws = x[:, z * each:(z + 1) * each], w[:, z * each:(z + 1) * each]
        assert ((parts[z].double() - xs.double() @ ws.double().T).abs() <= bound(xs, ws, each)).all()


@pytest.mark.parametrize("M", [17, 33, 64])
@pytest.mark.parametrize("N,K", [(32768, 1024), (40000, 264), (51201, 128), (24580, 320)])
def test_a_bias_on_uncut_tiles(M, N, K):
    """In the short end, where rows start at whole pieces, and in the other: off them by the stride, by N, by the result's address."""
    x, w, g = operands(M, N, K, M + N)
    biases = torch.randn(N + 1, device=DEV, generator=g).to(torch.bfloat16)
    ref, err = x.double() @ w.double().T, bound(x, w, K)
    for kind, ulp in ((torch.float32, 2.0 ** -23), (torch.bfloat16, 2.0 ** -8)):
        for wide, first in ((N + 8, 0), (N + 3, 0), (N + 8, 1)):
            bias = biases[first:first + N]                  # its address is off whole pieces too
            buf = torch.full((M, wide), float("nan"), device=DEV, dtype=kind)
            out = buf[:, first:first + N]
            ops()._few_rows("linear output", x, w, bias, out, 0, M, N, K, True)
            want = ref + bias.double()
            assert ((out.double() - want).abs() <= err + want.abs() * ulp).all()
            assert torch.isnan(buf[:, :first]).all() and torch.isnan(buf[:, first + N:]).all()
