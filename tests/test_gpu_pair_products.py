"""A wide product with a narrow float one beside it in one launch, and an expert layer's choice with the activation it weighs in one
kernel: the bits of the separate calls, over sizes on both sides of every line."""
import pytest
import torch

from reinfer_amd import kernels

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# rows of each form and past them; runs of 64 and of 128 k, k in no whole runs and past 8192, where walks start apart; features of less
# than a tile, of fewer tiles than workgroups, of more (walks start apart), off the tiles
@pytest.mark.parametrize("M", [1, 4, 5, 8, 9, 16, 17])
@pytest.mark.parametrize("N,N2,K", [(24, 1, 64), (6144, 32, 2560), (12288, 32, 4096), (8200, 17, 1032), (8176, 16, 4096), (512, 300, 8200),
                                    (9000, 48, 8712)])
def test_pair_has_the_bits_of_two_products(library_calls, M, N, N2, K):
    ops = kernels.current()
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K + 8, generator=g, device=DEV).bfloat16()[:, :K]
    w, w2 = (torch.randn(n, K, generator=g, device=DEV).bfloat16() * 0.02 for n in (N, N2))
    wide, narrow = torch.full((M, N + 8), 7.0, device=DEV, dtype=torch.bfloat16), torch.full((M, N2 + 3), 7.0, device=DEV)
    names = library_calls(lambda: ops.linear_pair(x, w, wide[:, :N], w2, narrow[:, :N2]))
    assert names == ["ra_gemm_skinny_pair"] if M <= 16 else "ra_gemm_skinny_pair" not in names
    one, two = torch.empty(M, N, device=DEV, dtype=torch.bfloat16), torch.empty(M, N2, device=DEV)
    ops.linear(x, w, one)
    ops.linear(x, w2, two)
    assert torch.equal(wide[:, :N], one) and torch.equal(narrow[:, :N2], two)
    assert (wide[:, N:] == 7.0).all() and (narrow[:, N2:] == 7.0).all()
    want = x.double() @ w2.double().t()
    assert ((two.double() - want).abs() <= (K + 2) * 2.0 ** -24 * (x.double().abs() @ w2.double().abs().t())).all()


def test_pairs_that_are_refused():
    ops = kernels.current()
    x, w = torch.zeros(4, 64, device=DEV, dtype=torch.bfloat16), torch.zeros(32, 64, device=DEV, dtype=torch.bfloat16)
    out, out2 = torch.empty(4, 32, device=DEV, dtype=torch.bfloat16), torch.empty(4, 32, device=DEV)
    for bad in (dict(weight=w[:, :32]), dict(weight2=w[:16]), dict(out2=out2[:2]), dict(out=out[:, :16])):
        args = dict(weight=w, out=out, weight2=w, out2=out2)
        args.update(bad)
        with pytest.raises(ValueError):
            ops.linear_pair(x, **args)


@pytest.mark.parametrize("T", [1, 8, 65])
@pytest.mark.parametrize("E,top,ff,shared,groups,kept", [(16, 4, 1024, 2048, 4, 2), (8, 2, 72, 0, 1, 1), (5, 5, 8, 24, 1, 1), (128, 8, 16, 8, 8, 3),
                                                         (6, 2, 12, 4, 2, 1), (70, 64, 8, 0, 1, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_choice_with_gated_experts(library_calls, T, E, top, ff, shared, groups, kept, dtype):
    ops = kernels.current()
    g = torch.Generator(device=DEV).manual_seed(T + E + ff)
    n = E * ff + shared
    up = (torch.randn(T, 2 * n, generator=g, device=DEV) * 2).to(dtype)
    logits = torch.randn(T, E + 3, generator=g, device=DEV)[:, :E]
    logits[0, : E // 2] = logits[0, 0]                                # ties
    if T > 1:
        logits[1, 1], logits[1, 2] = float("inf"), float("-inf")      # scores of one and zero
    act, want = torch.full((T, n), 7.0, device=DEV, dtype=dtype), torch.empty(T, n, device=DEV, dtype=dtype)
    choice = dict(scale=2.5, groups=groups, groups_kept=kept, group_top=2)
    names = library_calls(lambda: ops.moe_choose_scale(up, act, logits, top, E, ff, shared=shared, scoring="sigmoid", **choice))
    assert (names == ["ra_moe_choose_scale"]) == (ff % 8 == 0 and shared % 8 == 0)
    ids, weights = torch.empty(T, top, device=DEV, dtype=torch.int32), torch.empty(T, top, device=DEV)
    kernels.library.call("ra_moe_route_sigmoid", logits.data_ptr(), logits.stride(0), E, top, groups, kept, 2, 2.5, ids.data_ptr(),
                         weights.data_ptr(), T, torch.cuda.current_stream().cuda_stream)
    ops.moe_silu_gate_scale(up, want, ids, weights, E, ff, shared)
    assert torch.equal(act, want)
    score = torch.sigmoid(logits.double())
    assert torch.equal(score.gather(1, ids.long()).float(), (weights.double() / 2.5).float()) or \
        (score.gather(1, ids.long()) - weights.double() / 2.5).abs().max() < 1e-6


@pytest.mark.parametrize("T", [1, 8, 65])
@pytest.mark.parametrize("E,top,ff", [(16, 4, 1536), (3, 1, 8), (64, 6, 40), (10, 10, 12)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_choice_with_squared_experts(library_calls, T, E, top, ff, dtype):
    ops = kernels.current()
    g = torch.Generator(device=DEV).manual_seed(T + E + ff)
    up = (torch.randn(T, E * ff, generator=g, device=DEV) * 2).to(dtype)
    x, router = torch.randn(T, 64, generator=g, device=DEV).to(dtype), torch.randn(E, 64, generator=g, device=DEV).to(dtype)
    ids, weights = torch.empty(T, top, device=DEV, dtype=torch.int32), torch.empty(T, top, device=DEV)
    logits = ops.moe_route(x, router, top, ids, weights)
    act, want = torch.full((T, E * ff), 7.0, device=DEV, dtype=dtype), torch.empty(T, E * ff, device=DEV, dtype=dtype)
    names = library_calls(lambda: ops.moe_choose_scale(up, act, logits, top, E, ff))
    assert (names == ["ra_moe_choose_scale"]) == (ff % 8 == 0)
    ops.moe_relu2_scale(up, want, ids, weights, E, ff)
    assert torch.equal(act, want)
