"""The filters' boundaries where their slices, bins and lists end, against the plain chain."""
import pytest
import torch

import plain_qwen3 as plain

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def filtered(rows, params):
    from reinfer_amd import kernels
    from reinfer_amd.sampling import SamplingParams
    logits = torch.stack(rows).to(DEV)
    kernels.current().filter_logits(logits, [SamplingParams(**p) for p in params], [[1, 2, 3]] * len(rows))
    return logits.cpu()


FILTERS = [dict(temperature=0.7, top_k=1), dict(temperature=1.0, top_k=300), dict(temperature=0.9, top_p=0.9),
           dict(temperature=1.0, top_k=40, top_p=0.7), dict(temperature=1.2, top_k=2000, top_p=0.99, min_p=1e-3),
           dict(temperature=0.5, min_p=0.2), dict(temperature=1.0, top_k=10 ** 6), dict(temperature=1.0)]


@pytest.mark.parametrize("V", [1, 63, 4095, 4096, 4097, 12289])
@pytest.mark.parametrize("spread", [0.01, 1.0, 40.0])     # one bin, a bell over many, most beyond the last
def test_filters_at_the_edges_of_slices_and_bins(V, spread):
    g = torch.Generator().manual_seed(V)
    # values a clear step apart, in a random order: no boundary hangs on the last bit
    row = (torch.linspace(-3.0, 3.0, V) * spread)[torch.randperm(V, generator=g)]
    got = filtered([row] * len(FILTERS), FILTERS)
    for i, f in enumerate(FILTERS):
        kw = {k: v for k, v in f.items() if k != "temperature"}
        kept = torch.isfinite(plain.filter_logits(row, f["temperature"], **kw))
        mine = torch.isfinite(got[i])
        assert torch.equal(got[i][mine], row[mine])
        if f.get("top_p") and spread < 1.0:
            # neighbours' shares of the mass differ by less than the rounding of their exponentials (a few units of 2^-24
            # each): the boundary may lie that share of the row further
            assert abs(int(mine.sum()) - int(kept.sum())) <= 1 + V * 2.0 ** -20, (i, int(mine.sum()), int(kept.sum()))
            assert row[mine].min() > row[~mine].max() if (~mine).any() else True
        else:
            assert torch.equal(kept, mine), (i, int(kept.sum()), int(mine.sum()))


def test_filters_over_equal_logits_and_rows_with_few_finite_ones():
    V = 10000
    equal = torch.full((V,), 1.5)
    few = torch.full((V,), float("-inf"))
    few[[7, 4096, 9999]] = torch.tensor([1.0, 3.0, 2.0])
    few[11] = float("nan")
    none = torch.full((V,), float("nan"))
    got = filtered([equal, equal, few, few, none],
                   [dict(temperature=1.0, top_k=5000), dict(temperature=1.0, top_p=0.4), dict(temperature=1.0, top_k=2),
                    dict(temperature=1.0, top_k=50, top_p=0.6), dict(temperature=1.0, top_k=3, top_p=0.5)])
    assert torch.isfinite(got[0]).nonzero()[:, 0].tolist() == list(range(5000))      # the lower id first among equals
    assert torch.isfinite(got[1]).all()                                              # ties at the boundary all stay
    assert torch.isfinite(got[2]).nonzero()[:, 0].tolist() == [4096, 9999]
    assert torch.isfinite(got[3]).nonzero()[:, 0].tolist() == [4096]                 # 0.67 of the mass
    assert not torch.isfinite(got[4]).any()


@pytest.mark.parametrize("given", [0, 1, 2])
def test_rows_without_options_or_tokens_stay_as_they_are(given):
    """Fewer options, or fewer token lists, than rows: the rows behind them keep their logits."""
    from reinfer_amd import kernels
    from reinfer_amd.sampling import SamplingParams
    row = torch.linspace(-3.0, 3.0, 500)
    p = SamplingParams(temperature=1.0, top_k=7)
    for params, histories in (([p] * given, [[1, 2]] * 3), ([p] * 3, [[1, 2]] * given)):
        logits = torch.stack([row] * 3).to(DEV)
        kernels.current().filter_logits(logits, params, histories)
        kept = torch.isfinite(logits).sum(-1).tolist()
        assert kept == [7] * given + [500] * (3 - given)


def test_tokens_of_other_number_kinds():
    """Histories that hold numpy numbers, floats among them, count as the whole numbers that they are."""
    import numpy as np
    from reinfer_amd import kernels
    from reinfer_amd.sampling import SamplingParams
    p = [SamplingParams(temperature=1.0, presence_penalty=2.0)]
    want = None
    for history in ([3, 5], np.array([3, 5]), np.array([3.0, 5.0]), torch.tensor([3, 5]), (3, 5)):
        logits = torch.zeros(1, 16, device=DEV)
        kernels.current().filter_logits(logits, p, [history])
        want = logits.clone() if want is None else want
        assert torch.equal(logits, want) and logits[0, 3] == -2.0 and logits[0, 4] == 0.0


@pytest.mark.parametrize("window", [1, 255, 257, 1024, 1025, 3000])
@pytest.mark.parametrize("pad", [0, 3])
@pytest.mark.parametrize("bias", [(), ((3, 1.0), (4097, -2.0), (12288, 0.5))])
def test_penalties_over_windows_of_every_length(window, pad, bias):
    """Windows that are counted in LDS and longer ones, shorter and longer than a workgroup, with tokens on both sides of the
    window's start and in every slice; rows on 16 bytes and off. All numbers are exact in binary: so is the result."""
    from reinfer_amd import kernels
    from reinfer_amd.sampling import SamplingParams
    V = 12289
    g = torch.Generator().manual_seed(window)
    rows = torch.randint(-64, 64, (4, V), generator=g) / 16.0
    rows[:, [5, 9000]] = float("-inf")
    kinds = [dict(frequency_penalty=0.25), dict(repeat_penalty=2.0, presence_penalty=0.5),
             dict(temperature=1.0, top_k=40, repeat_penalty=4.0, frequency_penalty=0.125), dict(presence_penalty=0.5)]
    # few different tokens, so that they come again across the window's start; the last row's are all one
    histories = [torch.randint(0, 400, (3100,), generator=g).mul(V // 400).tolist() for _ in kinds[:3]] + [[12288] * 3100]
    params = [SamplingParams(repeat_last_n=window, logit_bias=bias, **k) for k in kinds]
    logits = torch.full((4, V + pad), 7.0, device=DEV)
    logits[:, :V] = rows.to(DEV)
    kernels.current().filter_logits(logits[:, :V], params, histories)
    got = logits.cpu()
    assert (got[:, V:] == 7.0).all()
    for i, k in enumerate(kinds):
        kw = {a: b for a, b in k.items() if a != "temperature"}
        want = plain.filter_logits(rows[i], k.get("temperature", 0.0), window=histories[i][-window:], logit_bias=bias, **kw)
        assert torch.equal(got[i, :V].double(), want), (i, (got[i, :V] != want).nonzero()[:5])
