"""The bfloat16 product of many rows against float64: every tile at its edges, with each epilogue, in K ranges, and its rule."""
import math

import pytest
import torch

from reinfer_amd import kernels

import test_gpu_moe_grouped as grouped

pytestmark = pytest.mark.gpu
DEV = "cuda"
TILES = [(m, n) for n in (256, 128) for m in (256, 224, 192, 160, 128)]


def ops():
    return kernels.current()


def operands(M, N, K, seed, stride=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K + stride, device=DEV, generator=g).to(torch.bfloat16)[:, :K]
    w = (torch.randn(N, K, device=DEV, generator=g) / math.sqrt(K)).to(torch.bfloat16)
    return x, w, g


def bound(x, w, K):
    """Float sums of K exact products in any order: K roundings of at most 2^-24 of the sum of magnitudes, which the
    matrix cores' own order halves many times over; a twentieth of that worst case still catches a lost or doubled k."""
    return (x.double().abs() @ w.double().abs().T) * (K * 2.0 ** -24 / 20) + 1e-6


def gated(prod, err):
    rows = torch.arange(prod.shape[1], device=DEV).view(-1, 2, 8)
    gate, up = prod[:, rows[:, 0].reshape(-1)], prod[:, rows[:, 1].reshape(-1)]
    eg, eu = err[:, rows[:, 0].reshape(-1)], err[:, rows[:, 1].reshape(-1)]
    want = gate * torch.sigmoid(gate) * up              # silu's slope is at most 1.1
    return want, 1.1 * eg * (up.abs() + eu) + gate.abs() * eu + want.abs() * (2 ** -8 + 2 ** -20)


# one row and one run of weight rows; a row less and more than tiles of every height, the least K; weight rows that end inside a
# tile; more tiles than workgroups, so that one takes several (five rows of 128 x 128 tiles in 66 columns)
SIZES = [(1, 16, 256), (129, 1040, 256), (255, 528, 320), (449, 272, 4096), (600, 8432, 384)]


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K", SIZES)
def test_every_tile_with_each_epilogue(M, N, K, tile):
    x, w, g = operands(M, N, K, M + N, stride=8)
    ref, err = x.double() @ w.double().T, bound(x, w, K)
    buf = torch.full((M + 1, N + 8), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops()._prompt(0, x, w, buf[:M, :N], tile=tile)
    assert ((buf[:M, :N].double() - ref).abs() <= err + ref.abs() * 2 ** -8).all()
    assert torch.isnan(buf[M]).all() and torch.isnan(buf[:, N:]).all()
    buf = torch.full((M + 1, N // 2 + 8), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops()._prompt(1, x, w, buf[:M, :N // 2], tile=tile)
    want, tol = gated(ref, err)
    assert ((buf[:M, :N // 2].double() - want).abs() <= tol).all()
    assert torch.isnan(buf[M]).all() and torch.isnan(buf[:, N // 2:]).all()
    stream = torch.randn(M + 1, N + 8, device=DEV, generator=g) * 8
    was, want = stream.clone(), stream[:M, :N].double() + 0.25 * ref
    ops()._prompt(2, x, w, stream[:M, :N], alpha=0.25, tile=tile)
    assert ((stream[:M, :N].double() - want).abs() <= err + want.abs() * 2 ** -23).all()
    assert torch.equal(stream[M], was[M]) and torch.equal(stream[:, N:], was[:, N:])
    buf = torch.full((M + 1, N + 8), float("nan"), device=DEV)
    ops()._prompt(3, x, w, buf[:M, :N], tile=tile)
    assert ((buf[:M, :N].double() - ref).abs() <= err).all()
    assert torch.isnan(buf[M]).all() and torch.isnan(buf[:, N:]).all()


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("M,N,K,ranges", [(300, 1040, 1024, 4), (129, 2064, 832, 2), (513, 4112, 2560, 3), (70, 16384, 512, 2)])
def test_ranges_get_a_plane_each(M, N, K, ranges, tile):
    """Ranges of the least steps and of unlike numbers of steps."""
    x, w, _ = operands(M, N, K, M + N)
    planes = torch.full((ranges, M, N), float("nan"), device=DEV)
    ops()._prompt(3, x, w, planes, tile=tile, ranges=ranges)
    k = -(-K // 64 // ranges) * 64
    for z in range(ranges):
        a, b = x[:, z * k:(z + 1) * k], w[:, z * k:(z + 1) * k]
        assert ((planes[z].double() - a.double() @ b.double().T).abs() <= bound(a, b, k)).all()


@pytest.mark.parametrize("M,N,K", [(129, 4096, 1024), (300, 2560, 9728), (700, 2560, 4096), (1024, 2560, 9728), (3072, 1024, 4096),
                                   (3073, 1024, 4096), (700, 4096, 1032), (700, 1048, 4096)])
def test_calls_that_may_take_it(M, N, K):
    """The entry points on both sides of the rule (rows, K in steps of 64, weight rows in runs of 16) and for rows that cannot be
    read in 16-byte pieces."""
    x, w, g = operands(M, N, K, M)
    ref, err = x.double() @ w.double().T, bound(x, w, K)
    odd = torch.empty(M, K + 12, device=DEV, dtype=torch.bfloat16)[:, 1:K + 1]
    odd.copy_(x)
    for a in (x, odd):
        out = torch.full((M, N), float("nan"), device=DEV, dtype=torch.bfloat16)
        ops().linear(a, w, out)
        assert ((out.double() - ref).abs() <= err + ref.abs() * 2 ** -8).all()
        for alpha in (1.0, 0.5):
            stream = torch.randn(M, N, device=DEV, generator=g)
            want = stream.double() + alpha * ref
            ops().linear_skinny(a, w, stream, accumulate=True, alpha=alpha)
            assert ((stream.double() - want).abs() <= err + want.abs() * 2 ** -23).all()
        if N % 16 == 0:
            out = torch.full((M, N // 2), float("nan"), device=DEV, dtype=torch.bfloat16)
            ops().gated_linear(a, w, out)
            want, tol = gated(ref, err)
            # the library's product is rounded before its gate
            tol = tol + (want.abs() + ref.abs().amax() * 0.1) * 2 ** -7
            assert ((out.double() - want).abs() <= tol).all()


@pytest.mark.parametrize("N,K", [(4096, 4096), (2560, 9728)])
def test_a_row_s_sums_do_not_depend_on_the_rows_beside_it(N, K):
    """Products that add into the stream, on both sides of where they become this kernel's."""
    x, w, g = operands(1500, N, K, N)
    stream = torch.randn(1500, N, device=DEV, generator=g)
    full = stream.clone()
    ops().linear_skinny(x, w, full, accumulate=True)
    for M in (600, 1024, 1301):
        part = stream[:M].clone()
        ops().linear_skinny(x[:M], w, part, accumulate=True)
        assert torch.equal(part, full[:M])


def test_a_row_s_sums_do_not_depend_on_the_tile():
    x, w, _ = operands(600, 1040, 2560, 5)
    outs = []
    for tile in TILES:
        outs.append(torch.empty(600, 1040, device=DEV))
        ops()._prompt(3, x, w, outs[-1], tile=tile)
    assert all(torch.equal(o, outs[0]) for o in outs)


def test_what_it_refuses():
    """Sizes that it cannot read or cut are errors of the library, not launches."""
    M, N, K = 256, 1040, 1024
    x, w, _ = operands(M, N, K, 1)
    out = torch.zeros(M, N, device=DEV)
    for args in [dict(tile=(96, 128)), dict(ranges=0), dict(ranges=2), dict(ranges=5), dict(ranges=17)]:
        with pytest.raises(kernels.KernelLibraryError):
            ops()._prompt(2, x, w, out, **args)
    for n, k in [(1048, 1024), (1040, 1000), (1040, 192)]:
        with pytest.raises(kernels.KernelLibraryError):
            ops()._prompt(3, x[:, :k], w[:min(n, N), :k].contiguous() if n <= N else torch.zeros(n, k, device=DEV, dtype=torch.bfloat16),
                          torch.zeros(M, n, device=DEV))
    assert out.abs().max() == 0


@pytest.mark.parametrize("M", [17, 48, 64])
@pytest.mark.parametrize("N,K", [(6144, 2560), (1536, 1024), (4096, 2552), (5120, 2048), (4099, 4096)])
def test_small_products_are_left_in_ranges(M, N, K):
    """From 10 M weights on; below, where the kernel whose waves split K takes them, the whole product is the faster one."""
    x, w, _ = operands(M, N, K, M + N)
    parts = ops().linear_ranges(x, w)
    if N * K < 10 << 20 and not kernels.library.load().ra_gemm_wide_preferred(0, M, N, K):
        assert parts is None
        return
    assert parts.shape[0] == kernels.library.load().ra_gemm_wide_ranges(M, N, K) >= 2
    assert ((parts.double().sum(0) - x.double() @ w.double().T).abs() <= bound(x, w, K)).all()


# experts in whole steps of 64: pairs of an expert on both sides of every tile height (128, 192 and 256 by the mean), experts without
# pairs, weight rows that end inside a tile (320 and 576 columns), both tile widths; the least widths
@pytest.mark.parametrize("T,E,top,ff,width", [(129, 3, 1, 256, 256), (100, 5, 2, 320, 576), (575, 9, 3, 320, 1088),
                                              (640, 3, 1, 576, 320), (1500, 16, 4, 1024, 512), (3000, 5, 2, 256, 2112)])
@pytest.mark.parametrize("gated_kind", [False, True])
@pytest.mark.parametrize("kind", ["spread", "one", "identity"])
def test_experts_in_whole_steps(T, E, top, ff, width, gated_kind, kind):
    grouped.test_experts_over_sorted_tokens(T, E, top, ff, width, gated_kind, kind)


@pytest.mark.parametrize("N,K", [(2560, 9728), (4096, 4096), (4096, 12288), (5120, 8192), (5120, 25600)])
def test_products_cut_into_ranges_have_one_order_of_sums_a_row_of_tiles(N, K):
    """129 to 256 rows (and the rows of further 128) share their ranges: a row's sums do not depend on the rows beside it. What is
    not cut at these rows is the library's, here in one chain."""
    x, w, g = operands(512, N, K, N + K)
    stream = torch.randn(512, N, device=DEV, generator=g)
    wq = w[:, :4096].repeat(3, 1)[:6144].contiguous()
    for sizes in [(129, 150, 160, 161, 193, 240, 256), (257, 300, 321, 384), (385, 448, 481, 482, 512)]:
        if kernels.library.load().ra_gemm_tile_takes(2, sizes[-1], N, K):
            outs = []
            for M in sizes:
                outs.append(stream[:M].clone())
                ops().linear_skinny(x[:M], w, outs[-1], accumulate=True)
            assert all(torch.equal(o[:sizes[0]], outs[0]) for o in outs)
        parts = [ops().linear_ranges(x[:M, :4096], wq) for M in sizes]
        assert len({p is None for p in parts}) == 1
        if parts[0] is not None:
            assert all(p.shape[0] == parts[0].shape[0] and torch.equal(p[:, :sizes[0]], parts[0]) for p in parts)


@pytest.mark.parametrize("M", [17, 64, 129])
def test_rows_off_16_bytes_are_not_left_in_ranges(M):
    """They are declined, as any product that the range kernels cannot read: the caller then asks for the whole product."""
    N, K = 6144, 4096
    x, w, _ = operands(M, N, K, M)
    buf = torch.empty(M * (K + 8) + 4, device=DEV, dtype=torch.bfloat16)[4:].view(M, K + 8)[:, :K]
    buf.copy_(x)
    wide = torch.empty(N * K + 4, device=DEV, dtype=torch.bfloat16)[4:].view(N, K)
    wide.copy_(w)
    same = x[:1].expand(M, K)                  # one row M times: a stride below K
    assert ops().linear_ranges(x, w) is not None
    assert all(ops().linear_ranges(a, b) is None for a, b in ((buf, w), (x, wide), (same, w)))


# both sides of every line of the rule: half of the chip's 256 CUs in tiles of 128 x 128, three quarters for plain products of a long K;
# plain ones whose 256 x 256 tiles fill their rounds, without padding; rows that fill every tile, or not, of one that adds
@pytest.mark.parametrize("epilogue,M,N,K,own", [
    (1, 129, 2048, 4096, False), (1, 512, 4096, 2560, False), (1, 513, 4096, 2560, True), (1, 256, 8192, 2048, True),
    (0, 768, 4096, 4096, False), (0, 769, 4096, 4096, True), (0, 513, 1024, 8192, False), (0, 1024, 2048, 2048, False),
    (0, 1025, 2048, 2048, True), (2, 1024, 2048, 2560, False), (2, 3072, 2048, 4096, True),
    (0, 3841, 4096, 2560, False), (0, 3840, 4096, 2560, True), (0, 4097, 4096, 2560, True), (0, 4096, 4112, 2560, True),
    (2, 768, 4096, 4096, False), (2, 700, 4096, 4096, True)])
def test_who_takes_a_product_of_many_rows(epilogue, M, N, K, own, monkeypatch):
    x, w, g = operands(M, N, K, M + N)
    ref, err = x.double() @ w.double().T, bound(x, w, K)
    calls, call = [], kernels.library.call
    monkeypatch.setattr(kernels.library, "call", lambda name, *a: (calls.append(name), call(name, *a))[1])
    if epilogue == 0:
        out = torch.full((M, N), float("nan"), device=DEV, dtype=torch.bfloat16)
        ops().linear(x, w, out)
        assert ((out.double() - ref).abs() <= err + ref.abs() * 2 ** -8).all()
    elif epilogue == 2:
        stream = torch.randn(M, N, device=DEV, generator=g)
        want = stream.double() + ref
        ops().linear_skinny(x, w, stream, accumulate=True)
        assert ((stream.double() - want).abs() <= err + want.abs() * 2 ** -23).all()
    else:
        want, tol = gated(ref, err)                     # neither way rounds gate and up
        for pad in (0, 8):
            buf = torch.full((M + 1, N // 2 + pad), float("nan"), device=DEV, dtype=torch.bfloat16)
            ops().gated_linear(x, w, buf[:M, :N // 2])
            assert ((buf[:M, :N // 2].double() - want).abs() <= tol).all()
            assert torch.isnan(buf[M]).all() and torch.isnan(buf[:, N // 2:]).all()
            if pad == 0:
                assert ("ra_silu_mul_rounded" in calls) != own
        return
    assert ("ra_gemm_prompt" in calls) == own


# 16 MB of experts: one tile an expert by the mean, where their weights are read past the caches, and two; with all tokens at one
# expert ("one") more than the mean says
@pytest.mark.parametrize("T,E,top,ff,width", [(300, 16, 4, 512, 1024), (1100, 16, 4, 512, 1024)])
@pytest.mark.parametrize("gated_kind", [False, True])
@pytest.mark.parametrize("kind", ["spread", "one"])
def test_experts_of_one_tile_each(T, E, top, ff, width, gated_kind, kind):
    grouped.test_experts_over_sorted_tokens(T, E, top, ff, width, gated_kind, kind)
