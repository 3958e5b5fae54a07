"""Experts over sorted tokens against a plain sum over every token's choices."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def ops():
    from reinfer_amd import kernels
    return kernels.current()


def choices(kind, T, E, top, g):
    if kind == "spread":
        return torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)])
    if kind == "one":                        # every token the same experts, the others none: full tiles and empty experts
        return torch.arange(top).expand(T, top).clone()
    ids = torch.stack([torch.randperm(E + 2, generator=g)[:top] for _ in range(T)])      # "identity": ids past the experts
    ids[0] = E
    return ids


# slots of an expert on both sides of a tile of 128; k and weight rows that end inside a step and a tile, rows in steps of
# 8 alone; both tile widths (256 needs two tiles a CU)
@pytest.mark.parametrize("T,E,top,ff,width", [(65, 5, 2, 40, 72), (127, 3, 1, 64, 128), (128, 3, 1, 72, 264),
                                              (129, 3, 1, 136, 64), (400, 9, 3, 24, 200), (1500, 16, 4, 264, 4104)])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("kind", ["spread", "one", "identity"])
def test_experts_over_sorted_tokens(T, E, top, ff, width, gated, kind):
    g = torch.Generator().manual_seed(T + ff)
    G = torch.Generator(device=DEV).manual_seed(T + ff)
    shared = 16
    x = torch.randn(T, width + 8, generator=G, device=DEV).bfloat16()[:, :width]
    n_up = 2 if gated else 1
    w_up = (torch.randn(n_up * (E * ff + shared), width, generator=G, device=DEV) / width ** 0.5).bfloat16()
    w_down = (torch.randn(width, E * ff + shared, generator=G, device=DEV) / ff ** 0.5).bfloat16()
    ids = choices(kind, T, E, top, g).to(torch.int32).to(DEV).contiguous()
    wts = torch.rand(T, top, generator=G, device=DEV)
    more = torch.randn(T, width, generator=G, device=DEV) if gated else None
    logit = torch.randn(T, 3, generator=G, device=DEV)[:, 1] if gated else None
    assert top > 0.4 * E or ops().moe_groups(x, w_up, w_down, top, E, ff)
    want = torch.zeros(T, width, dtype=torch.float64, device=DEV)
    size = torch.zeros_like(want)            # of the terms, for the bound
    xd = x.double()
    for e in range(E):
        rows = (ids == e).any(-1).nonzero()[:, 0]
        p = (wts * (ids == e)).sum(-1)[rows, None].double()
        u = w_up[n_up * e * ff:n_up * (e + 1) * ff].double()
        a = torch.nn.functional.silu(xd[rows] @ u[:ff].t()) * (xd[rows] @ u[ff:].t()) if gated else \
            torch.relu(xd[rows] @ u.t()) ** 2
        d = w_down[:, e * ff:(e + 1) * ff].double().t()
        want[rows] += (p * a) @ d
        size[rows] += (p * a).abs() @ d.abs()
    same = (wts * (ids >= E)).sum(-1, keepdim=True).double()
    want += same * xd
    size += same * xd.abs()
    if more is not None:
        want += more.double() * torch.sigmoid(logit[:, None].double())
    # the activation is rounded once to bfloat16 (2^-9 of each term at most); float sums stay far below that
    bound = 2.0 ** -8 * size + 1e-4
    out = torch.full((T, width), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops().moe_grouped(x, w_up, w_down, ids, wts, E, ff, gated, more=more, more_logit=logit, out=out)
    assert ((out.double() - want).abs() <= bound + 2.0 ** -8 * want.abs()).all()
    resid = torch.randn(T, width, generator=G, device=DEV)
    base = resid.double()
    ops().moe_grouped(x, w_up, w_down, ids, wts, E, ff, gated, more=more, more_logit=logit, resid=resid, alpha=0.5)
    assert ((resid.double() - (base + 0.5 * want)).abs() <= bound).all()


@pytest.mark.parametrize("T,E,top,ff,width", [(65, 8, 3, 40, 72), (300, 16, 4, 64, 128)])
def test_an_expert_that_a_token_names_twice(T, E, top, ff, width):
    """Its last weight counts, as in the products over all experts side by side."""
    g, G = torch.Generator().manual_seed(T), torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(T, width, generator=G, device=DEV).bfloat16()
    w_up = (torch.randn(2 * E * ff, width, generator=G, device=DEV) / width ** 0.5).bfloat16()
    w_down = (torch.randn(width, E * ff, generator=G, device=DEV) / ff ** 0.5).bfloat16()
    ids = choices("spread", T, E, top, g)
    ids[::3, 0] = ids[::3, top - 1]
    ids[1::3, 1] = ids[1::3, 0]
    ids[5] = ids[5, 0]
    ids = ids.to(torch.int32).to(DEV)
    wts = torch.rand(T, top, generator=G, device=DEV)
    gu, act = torch.empty(T, 2 * E * ff, device=DEV).bfloat16(), torch.empty(T, E * ff, device=DEV).bfloat16()
    ops().linear(x, w_up, gu)
    ops().moe_silu_gate_scale(gu, act, ids, wts, E, ff)
    want = act.double() @ w_down.double().t()
    size = act.double().abs() @ w_down.double().abs().t()
    out = torch.empty(T, width, dtype=torch.bfloat16, device=DEV)
    ops().moe_grouped(x, w_up, w_down, ids, wts, E, ff, True, out=out)
    # the products before the activation are rounded to bfloat16 on one side alone, the activations on both
    assert ((out.double() - want).abs() <= 2.0 ** -6 * size + 2.0 ** -8 * want.abs() + 1e-4).all()


def test_an_id_below_zero_names_nothing():
    T, E, top, ff, width = 70, 8, 3, 40, 72
    G = torch.Generator(device=DEV).manual_seed(T)
    x = torch.randn(T, width, generator=G, device=DEV).bfloat16()
    w_up = (torch.randn(E * ff, width, generator=G, device=DEV) / width ** 0.5).bfloat16()
    w_down = (torch.randn(width, E * ff, generator=G, device=DEV) / ff ** 0.5).bfloat16()
    ids = torch.arange(top, device=DEV, dtype=torch.int32).repeat(T, 1)
    wts = torch.rand(T, top, generator=G, device=DEV)
    wts[7, 0] = 0.0
    out, want = (torch.empty(T, width, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ops().moe_grouped(x, w_up, w_down, ids, wts, E, ff, False, out=want)
    ids[7, 0] = -5
    ops().moe_grouped(x, w_up, w_down, ids, wts, E, ff, False, out=out)
    assert torch.equal(out, want)


def test_where_sorting_pays():
    """Decode steps of up to 128 requests, and short steps beside a shared expert, stay with the products over all experts unless
    few are chosen."""
    pay = ops().moe_groups_pay
    assert not any(pay(T, 4, 16) or pay(T, 2, 8) for T in (65, 128)) and pay(129, 4, 16) and pay(1900, 4, 16)
    assert not pay(256, 4, 16, True) and pay(257, 4, 16, True)
    assert not pay(64, 6, 64) and pay(65, 6, 64) and pay(65, 8, 128)


def test_captured_steps_over_sorted_tokens(tmp_path):
    """A decode step of 70 requests whose tokens choose 2 of 32 experts: replays between other work against eager steps."""
    import json
    import os
    from helpers import random_tokens
    from kobolix_helpers import _dense, _memory, _moe, draw_weights
    from reinfer_amd.engine import ModelRunner, StepEntry
    from reinfer_amd.weights.safetensors_io import write_safetensors
    raw = {"architecture": "Kobolix", "vocab": 90, "width": 64, "norm": {"eps": 1e-5},
           "layers": [{"type": "mlstm", "mixer": _memory(2, 16, 24, 12.0), "mlp": _moe(32, 2, 24, shared=16)},
                      {"type": "mlstm", "mixer": _memory(1, 32, 16, 12.0), "mlp": _dense(40)}]}
    with open(os.path.join(str(tmp_path), "config.json"), "w") as f:
        json.dump(raw, f)
    write_safetensors(os.path.join(str(tmp_path), "model.safetensors"), draw_weights(raw, 5, torch.bfloat16), metadata={"format": "pt"})
    n, tokens = 70, random_tokens(70 * 8, 90, 3)
    found, calls = [], []
    kind = type(ops())
    real = kind.moe_grouped
    kind.moe_grouped = lambda *a, **k: (calls.append(1), real(*a, **k))[1]
    try:
        for graphs in (True, False):
            runner = ModelRunner.from_folder(str(tmp_path), dtype="bfloat16", device=DEV, max_seqs=n, max_model_len=64, use_graphs=graphs)
            out, seen = [], len(calls)
            for r in range(n):
                runner.add_request(r)
            for s in range(7):
                out.append(runner.step([StepEntry(r, [tokens[s * n + r]], [0]) for r in range(n)]).clone())
                torch.randn(500, 500, device=DEV).sum().item()
            assert len(calls) > seen
            found.append(out)
    finally:
        kind.moe_grouped = real
    for s, (a, b) in enumerate(zip(*found)):
        assert torch.isfinite(a).all() and torch.equal(a, b), s


def test_weights_are_held_once():
    from kobolix_helpers import _memory, _moe, draw_weights
    from reinfer_amd.config import config_from_dict
    from reinfer_amd.parts.moe import MixtureOfExperts
    raw = {"architecture": "Kobolix", "vocab": 90, "width": 64, "norm": {"eps": 1e-5},
           "layers": [{"type": "mlstm", "mixer": _memory(2, 16, 24, 12.0), "mlp": _moe(8, 2, 24, shared=16)}]}
    weights = {n: t.to(DEV) for n, t in draw_weights(raw, 5, torch.bfloat16).items() if ".mlp." in n}
    spec = config_from_dict(raw).to_spec().blocks[0].ffn
    part = MixtureOfExperts(spec, weights, "l0.mlp.", torch.bfloat16, torch.device(DEV))
    held = {t.untyped_storage().data_ptr(): t.untyped_storage().nbytes() for t in vars(part).values() if isinstance(t, torch.Tensor)}
    assert sum(held.values()) == sum(t.numel() * t.element_size() for t in weights.values())
