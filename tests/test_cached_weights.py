"""Models whose weights stay in the last-level cache from step to step: products read them by the caches' usual policy."""
import pytest
import torch

from helpers import TINY_A
from kernel_double import KernelDouble
from reinfer_amd import kernels
from reinfer_amd.config import config_from_dict
from reinfer_amd.engine import ModelRunner, StepEntry
from reinfer_amd.kernels import library
from reinfer_amd.kernels import ops as hip
from reinfer_amd.models import declare_params
from reinfer_amd.weights import random_tensors


class Scoped(KernelDouble):
    """Counts products inside and outside of ``cached_weights``."""
    def __init__(self, most):
        self.CACHED_WEIGHTS, self.depth, self.inside, self.outside = most, 0, 0, 0

    def cached_weights(self):
        return self

    def __enter__(self):
        self.depth += 1

    def __exit__(self, *_):
        self.depth -= 1

    def linear(self, *args):
        self.inside, self.outside = self.inside + (self.depth > 0), self.outside + (self.depth == 0)
        return super().linear(*args)


def step(raw, ops):
    cfg = config_from_dict(raw)
    weights = random_tensors(declare_params(cfg.to_spec()), 0, torch.float32)
    with kernels.use(ops):
        runner = ModelRunner.from_config(cfg, dtype="float32", device="cpu", weights=weights, max_tokens=64)
        runner.add_request("s")
        runner.step([StepEntry("s", [1, 2, 3], [2])])
    return runner.model.weight_bytes, weights


@pytest.mark.parametrize("tied", [False, True])
def test_a_model_of_at_most_the_cache_says_so(tied):
    raw = {**TINY_A, "tie_word_embeddings": tied}
    size, weights = step(raw, KernelDouble())
    embedding = next(t for n, t in weights.items() if "embed" in n).numel() * 4
    assert size == sum(t.numel() * 4 for n, t in weights.items() if not (tied and "lm_head" in n)) - (0 if tied else embedding)
    for most, all_inside in ((size, True), (size - 1, False)):
        ops = Scoped(most)
        step(raw, ops)
        assert ops.depth == 0 and (ops.outside == 0) == all_inside and (ops.inside > 0) == all_inside


@pytest.mark.gpu
def test_inside_every_product_keeps_to_the_usual_policy(monkeypatch):
    """The same bits from either instance of each kernel, and the hint in every call."""
    said, call = [], library.call
    monkeypatch.setattr(library, "call", lambda name, *args: (said.append((name, args[-2])), call(name, *args))[1])
    ops, dev, (N, K) = kernels.current(), "cuda:0", (4096, 2560)
    g = torch.Generator(device=dev).manual_seed(1)
    w = (torch.randn(N, K, device=dev, generator=g) * 0.02).bfloat16()
    w2 = (torch.randn(32, K, device=dev, generator=g) * 0.02).bfloat16()
    f = torch.randn(N, K, device=dev, generator=g) * 0.02
    up, down = (torch.randn(s, device=dev, generator=g).mul_(0.02).bfloat16() for s in ((16 * 512, 1024), (1024, 16 * 512)))

    def results(M):
        x = torch.randn(M, K, device=dev, generator=torch.Generator(device=dev).manual_seed(M))
        h, out = x.bfloat16(), []

        def new(*shape, dtype=torch.float32):
            out.append(torch.zeros(shape, device=dev, dtype=dtype))
            return out[-1]
        ss = torch.ones(1, M, device=dev)
        if M > 256:
            token = torch.arange(4, device=dev, dtype=torch.int32)
            ids = ((torch.arange(M, device=dev, dtype=torch.int32)[:, None] + token) % 16).contiguous()
            ops.moe_grouped(x[:, :1024].bfloat16().contiguous(), up, down, ids, torch.ones(M, 4, device=dev), experts=16, ff=512, gated=False,
                            out=new(M, 1024, dtype=torch.bfloat16))
            return out
        if M <= 16:
            ops.linear_pair(h, w, new(M, N, dtype=torch.bfloat16), w2, new(M, 32))
        if M <= 64:
            ops.linear(h, w, new(M, N))
            ops.linear_skinny(h, w, new(M, N), row_sums=(ss, 1e-6, K))
            ops.gated_linear(h, w, new(M, N // 2, dtype=torch.bfloat16))
            ops.linear(x, f, new(M, N))
            ops.linear_skinny(h, w, new(M, N), accumulate=True, alpha=0.5)
        ops.linear_skinny(h, w, new(M, N), accumulate=True)
        if M > 64 and ops.can_finish_norm(M, N, K):
            ops.linear_skinny(h, w, new(M, N), accumulate=True, finish=(torch.ones(N, device=dev), new(M, N, dtype=torch.bfloat16), 1e-6))
        parts = ops.linear_ranges(h, w) if M > 16 else None
        return out + ([parts] if parts is not None else [])

    for M in (1, 9, 17, 33, 64, 97, 300):
        said.clear()
        past = results(M)
        products = [n for n, _ in said if n.startswith(("ra_gemm_skinny", "ra_gemm_wide", "ra_gemm_f32", "ra_moe_grouped"))]
        assert products and all(k == 0 for n, k in said if n in products)
        said.clear()
        with hip.HipKernels.cached_weights():
            kept = results(M)
        assert [n for n, k in said if n in products] == products and all(k == 1 for n, k in said if n in products)
        assert len(past) == len(kept) and all(torch.equal(a, b) for a, b in zip(past, kept))
