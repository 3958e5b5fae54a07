"""Prompts of networks whose layers choose experts: products by the library, whose sums their routers have always decided by."""
import pytest
import torch

import detatar_helpers
import gibavik_helpers
import kobolix_helpers
import puresun_helpers
from helpers import TINY_A
from kernel_double import KernelDouble
from reinfer_amd import kernels
from reinfer_amd.config import config_from_dict
from reinfer_amd.engine import ModelRunner, StepEntry
from reinfer_amd.models import DecoderModel, declare_params
from reinfer_amd.weights import random_tensors

ROUTED = [kobolix_helpers, detatar_helpers, puresun_helpers]
# experts that a table gives by the token's number (gibavik) are nobody's choice
PLAIN = [gibavik_helpers]


def model(raw):
    spec = config_from_dict(raw).to_spec()
    return DecoderModel(spec, random_tensors(declare_params(spec), 1, torch.float32), torch.float32, torch.device("cpu"))


def chooses(raw):
    return any("router" in (layer.get("mlp") or {}) for layer in raw["layers"])


@pytest.mark.parametrize("helpers", ROUTED + PLAIN, ids=lambda h: h.__name__)
def test_who_asks_for_the_library(helpers):
    for raw, _ in helpers.CONFIGS.values():
        assert model(raw).routes == (helpers in ROUTED and chooses(raw))
    assert not model(TINY_A).routes


class Scoped(KernelDouble):
    """Counts calls inside and outside of ``library_products``."""
    def __init__(self):
        self.depth, self.inside, self.outside = 0, 0, 0

    def library_products(self):
        return self

    def __enter__(self):
        self.depth += 1

    def __exit__(self, *_):
        self.depth -= 1

    def linear(self, *args):
        self.inside, self.outside = self.inside + (self.depth > 0), self.outside + (self.depth == 0)
        return super().linear(*args)


@pytest.mark.parametrize("raw,routed", [(kobolix_helpers.KB_A, True), (TINY_A, False)], ids=["routed", "dense"])
def test_every_layer_s_products_stand_inside(raw, routed):
    ops = Scoped()
    with kernels.use(ops):
        runner = ModelRunner.from_config(config_from_dict(raw), dtype="float32", device="cpu", num_blocks=8,
                                         weights=random_tensors(declare_params(config_from_dict(raw).to_spec()), 2, torch.float32))
        runner.add_request("a")
        runner.step([StepEntry("a", [3, 1, 4], [2])])
    assert ops.depth == 0 and (ops.inside if routed else ops.outside) > 1
    assert ops.outside == 1 if routed else ops.inside == 0       # the head's product stands outside: its rows choose nothing


def test_the_scope_is_the_thread_s_own():
    import threading
    from reinfer_amd.kernels import ops
    seen = []
    with ops.HipKernels.library_products():
        t = threading.Thread(target=lambda: seen.append(getattr(ops._scope, "library", False)))
        t.start()
        t.join()
        with ops.HipKernels.library_products():
            pass
        assert ops._scope.library and seen == [False]
    assert not ops._scope.library


@pytest.mark.gpu
def test_products_inside_are_the_library_s():
    ops, dev = kernels.current(), "cuda"
    M, N, K = 700, 8192, 1024
    g = torch.Generator(device=dev).manual_seed(1)
    x = torch.randn(M, K, device=dev, generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, device=dev, generator=g) / 16).to(torch.bfloat16)
    stream = torch.randn(M, N, device=dev, generator=g)
    gu, want, out = (torch.empty(M, n, device=dev, dtype=torch.bfloat16) for n in (N, N // 2, N // 2))
    torch.mm(x, w.t(), out=gu)
    ops.silu_mul(gu, want, ops.GATE_GROUP)
    added = torch.addmm(stream, x, w.t(), out_dtype=torch.float32)
    with ops.library_products():
        ops.gated_linear(x, w, out)
        plain = torch.empty_like(gu)
        ops.linear(x, w, plain)
        ops.linear_skinny(x, w, stream, accumulate=True)
    assert torch.equal(out, want) and torch.equal(plain, gu) and torch.equal(stream, added)
    ops.gated_linear(x, w, out)
    assert not torch.equal(out, want)           # outside: gate and up are not rounded


@pytest.mark.gpu
def test_a_prompt_through_experts_has_the_library_s_bits(monkeypatch):
    h = kobolix_helpers
    raw = {"architecture": "Kobolix", "vocab": 512, "width": 1024, "norm": {"eps": 1e-6}, "residual_mult": 0.5,
           "embedding": {"scale": 4.0},
           "layers": [{"type": "mlstm", "mixer": h._memory(4, 128, 256, 15.0), "mlp": h._dense(4096)},
                      {"type": "parallel", "mixer": {"left": h._attn(8, 4, 128, 128, 64), "right": h._delta(8, 4, 128, 128, 4)},
                       "mlp": h._moe(8, 2, 512, groups=(4, 2), shared=1024)}]}
    cfg = config_from_dict(raw)
    weights = random_tensors(declare_params(cfg.to_spec()), 3, torch.bfloat16)
    calls = []
    call = kernels.library.call
    monkeypatch.setattr(kernels.library, "call", lambda name, *a: (calls.append(name), call(name, *a))[1])
    outs = []
    for taken in (True, False):
        if not taken:
            monkeypatch.setattr(type(kernels.current()), "_prompt_takes", classmethod(lambda *a: False))
        runner = ModelRunner.from_config(cfg, dtype="bfloat16", device="cuda:0", weights=weights, num_blocks=64, max_model_len=800)
        runner.add_request("a")
        outs.append(runner.step([StepEntry("a", [(7 * i) % 512 for i in range(700)], [0, 350, 699])]).clone())
    assert "ra_gemm_prompt" not in calls and len(calls) > 20
    assert torch.equal(outs[0], outs[1])
