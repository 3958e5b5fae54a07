"""Filters and draw in one go against the filter, then the draw: the same tokens, and the logits left as they are."""
import random

import pytest
import torch

from reinfer_amd import kernels
from reinfer_amd.sampling import Sampler, SamplingParams
from reinfer_amd.sampling.sampler import SamplingError, as_int64

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def two_steps(logits, params, seeds, positions, histories):
    """What the two kernels give one after the other."""
    ops = kernels.current()
    logits, n = logits.clone(), len(params)
    ops.filter_logits(logits, params, histories)
    tokens = torch.empty(n, dtype=torch.int32, device=DEV)
    ops.sample(logits, torch.tensor([max(0.0, p.temperature) for p in params], device=DEV), torch.tensor([as_int64(s) for s in seeds],
               device=DEV), torch.tensor(positions, dtype=torch.int32, device=DEV), tokens)
    return tokens.tolist()


def options(r, V, k):
    """Rows of every kind: none, each filter, each penalty, a bias, all together; greedy ones and drawn."""
    pick = lambda p, v: v if r.random() < p else None
    return SamplingParams(temperature=r.choice([0.0, 0.7, 1.0, 1.3]), top_k=pick(0.4, r.choice([1, 2, 50, V - 1, V])),
                          top_p=pick(0.4, r.choice([0.05, 0.9, 0.999])), min_p=pick(0.3, 0.05), repeat_penalty=pick(0.3, 1.2),
                          frequency_penalty=pick(0.3, 0.4), presence_penalty=pick(0.3, 0.5), repeat_last_n=r.choice([0, 1, 64, 1000, 4000]),
                          logit_bias=[(3, 4.0), (V - 1, -2.0)] if k % 5 == 4 else (), seed=r.getrandbits(60), max_tokens=4)


# less than a thread's four, a slice and more, off 16 bytes, the larger models'; windows of none to more than LDS holds
@pytest.mark.parametrize("V,stride", [(5, 5), (4096, 4096), (4097, 4099), (32768, 32768), (50003, 50004), (151936, 151936)])
@pytest.mark.parametrize("n", [1, 3, 24])
def test_same_tokens_as_filter_then_draw(library_calls, V, stride, n):
    r = random.Random(V + n)
    g = torch.Generator(device=DEV).manual_seed(V + n)
    logits = (torch.randn(n, stride, generator=g, device=DEV) * 3)[:, :V]
    if V > 5:
        logits[:, 7] = logits[:, 2]                                 # ties
        logits[0, V // 2:] = float("-inf")
        logits[n - 1, 1] = float("nan")
    before = logits.clone()
    for turn in range(6):
        params = [options(r, V, i + turn) for i in range(n)]
        histories = [[r.randrange(min(V, 40) if i % 2 else V) for _ in range(r.choice([0, 1, 64, 900, 3000]))] for i in range(n)]
        seeds, positions = [p.seed for p in params], [len(h) + 1 for h in histories]
        tokens = []
        names = library_calls(lambda: tokens.extend(Sampler(torch.device(DEV)).sample(logits, params, seeds, positions, histories)))
        assert names == ["ra_sample_filtered" if any(p.filters for p in params) else "ra_sample"]
        assert tokens == two_steps(logits, params, seeds, positions, histories), turn
        assert torch.equal(logits.view(torch.int32), before.view(torch.int32)) if stride == V else torch.equal(logits.nan_to_num(9), before.nan_to_num(9))


def test_a_row_without_a_finite_logit_and_rows_apart():
    logits = torch.randn(3, 2, 500, device=DEV)[:, 0]               # rows of 500, 1000 apart
    params = [SamplingParams(temperature=1.0, top_k=5, seed=1, max_tokens=2)] * 3
    args = (params, [1, 2, 3], [4, 5, 6], [[1], [2], [3]])
    assert Sampler(torch.device(DEV)).sample(logits, *args) == two_steps(logits, *args)
    every_second = torch.randn(3, 1000, device=DEV)[:, ::2]
    assert Sampler(torch.device(DEV)).sample(every_second, *args) == two_steps(every_second, *args)
    logits[1] = float("-inf")
    with pytest.raises(SamplingError, match="row 1"):
        Sampler(torch.device(DEV)).sample(logits, *args)
    # fewer histories than rows: the others' options are not applied, as ever
    short = ([params[0]] * 3, [1, 2, 3], [4, 5, 6], [[1]])
    assert Sampler(torch.device(DEV)).sample(every_second, *short) == two_steps(every_second, *short)
