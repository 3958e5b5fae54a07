"""The native packing of sampling options against the one in Python, over every kind of option and token that either takes."""
import random

import numpy as np
import pytest

from reinfer_amd._hostlib import host
from reinfer_amd.kernels.ops import HipKernels
from reinfer_amd.sampling import SamplingParams

general = HipKernels._pack_filters


def native(params, histories, n):
    packed = host.pack_filters(params, histories, n)
    return None if packed is None else np.frombuffer(packed, dtype=np.int32)


def test_random_options():
    r = random.Random(3)
    for _ in range(200):
        rows = r.randrange(1, 6)
        params = [SamplingParams(
            temperature=r.choice([0.0, -1.0, 0.7, 1e-40, float("inf")]), top_k=r.choice([None, 0, 50, 2 ** 31 - 1]),
            top_p=r.choice([None, 0.0, 0.9, 2.0]), min_p=r.choice([None, 0.05, -1.0]),
            repeat_penalty=r.choice([None, 0.5, 1.0, 1.1]), frequency_penalty=r.choice([None, -0.5, 0.1]),
            presence_penalty=r.choice([None, 0.0, 0.5, -2.0]), repeat_last_n=r.choice([0, 1, 5, 64])) for _ in range(rows)]
        histories = [[r.randrange(-2, 2 ** 31) for _ in range(r.choice([0, 1, 7, 100]))] for _ in range(rows)]
        n = rows + r.choice([0, 0, 2])                   # rows without options stay as they are
        assert np.array_equal(native(params, histories, n), general(params, histories, n))
        assert np.array_equal(native(tuple(params), histories[:1], n), general(params, histories[:1], n))
    assert np.array_equal(native([], [], 3), general([], [], 3))


@pytest.mark.parametrize("params,history", [
    (dict(temperature=1), [1]), (dict(temperature=np.float32(0.5)), [1]), (dict(temperature=0.5, top_p=1), [1]),
    (dict(top_k=np.int64(3)), [1]), (dict(top_k=True), [1]), (dict(logit_bias=((3, 1.0),)), [1]),
    (dict(repeat_penalty=1.2), (1, 2, 3)), (dict(repeat_penalty=1.2), np.arange(5)),
    (dict(repeat_penalty=1.2), [np.int64(7)]), (dict(repeat_penalty=1.2), [True]), (dict(repeat_penalty=1.2), [3.0])])
def test_other_kinds_go_the_general_way(params, history):
    p = [SamplingParams(**params)]
    assert native(p, [history], 1) is None
    assert general(p, [history], 1).dtype == np.int32


def test_what_neither_takes():
    many = [SamplingParams(), SamplingParams()]
    assert native(many, [[], []], 1) is None
    with pytest.raises(ValueError):
        general(many, [[], []], 1)
    big = [SamplingParams(top_k=2 ** 31)]
    assert native(big, [[]], 1) is None
    with pytest.raises(OverflowError):
        general(big, [[]], 1)
    far = [SamplingParams(repeat_penalty=1.2)]
    assert native(far, [[2 ** 31]], 1) is None


def test_options_without_a_bias_attribute():
    class Plain:
        temperature, top_k, top_p, min_p = 0.5, 3, None, None
        repeat_penalty, frequency_penalty, presence_penalty, repeat_last_n = 1.5, None, None, 2
    assert np.array_equal(native([Plain()], [[4, 5, 6]], 1), general([Plain()], [[4, 5, 6]], 1))
    with pytest.raises(AttributeError):
        native([object()], [[]], 1)
