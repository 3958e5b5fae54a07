"""Which form a recurrence takes, token by token or in chunks: what may depend on it and what may not."""
import json
import os

import pytest
import torch

from helpers import random_tokens, run_plan
from kobolix_helpers import _attn, _delta, _dense, _memory, draw_weights
from reinfer_amd import kernels
from reinfer_amd.engine import ModelRunner
from reinfer_amd.weights.safetensors_io import write_safetensors
from test_gpu_kobolix_kernels import DEV, make_batch

pytestmark = pytest.mark.gpu

MEMORIES = {"architecture": "Kobolix", "vocab": 90, "width": 64, "norm": {"eps": 1e-5},
            "layers": [{"type": "mlstm", "mixer": _memory(5, 64, 20, 12.0), "mlp": _dense(96)},
                       {"type": "parallel", "mixer": {"left": _attn(4, 2, 24, 16, 12), "right": _delta(4, 2, 20, 12, 3)},
                        "mlp": _dense(40)}]}


def runner_of(raw, folder, dtype):
    os.makedirs(folder)
    with open(os.path.join(folder, "config.json"), "w") as f:
        json.dump(raw, f)
    kind = torch.float32 if dtype == "float32" else torch.bfloat16
    write_safetensors(os.path.join(folder, "model.safetensors"), draw_weights(raw, 5, kind), metadata={"format": "pt"})
    return ModelRunner.from_folder(folder, dtype=dtype, device="cuda:0", max_tokens=8 * 192, max_seqs=8)


def test_32_bit_results_do_not_depend_on_the_requests_beside(tmp_path):
    """A request whose tokens come one to seven at a time, alone and beside a prompt in long portions."""
    runner = runner_of(MEMORIES, str(tmp_path / "m"), "float32")
    a, b = random_tokens(40, 90, 1), random_tokens(150, 90, 2)
    mine = [7, 1, 1, 16, 3, 1, 11]
    alone = run_plan(runner, {"a": a}, [[("a", n)] for n in mine])["a"]
    beside = run_plan(runner, {"a": a, "b": b}, [[("a", n), ("b", m)] for n, m in zip(mine, [17, 50, 1, 33, 16, 30, 3])])["a"]
    assert torch.equal(alone, beside)


@pytest.mark.parametrize("kind", ["memory", "delta"])
@pytest.mark.parametrize("mine,others", [(1, [64]), (16, [17]), (17, [1, 1]), (40, [3, 200]), (63, [64]), (64, [63, 1]), (100, [1, 65])])
def test_a_scan_does_not_depend_on_the_requests_beside(kind, mine, others):
    """bfloat16 rows, the form left to the call: a request's read-out and state alone and in the middle of a step."""
    ops = kernels.current()
    H, dk, dv = 3, 128, 40
    g = torch.Generator().manual_seed(mine)
    lens = [others[0], mine] + others[1:]
    T, at, width = sum(lens), others[0], 2 * H * dk + H * dv
    rows = (torch.randn(T, width, generator=g) * 0.3).to(torch.bfloat16).to(DEV)
    gates, bias = torch.randn(T, 2 * H, generator=g).to(DEV), torch.randn(2 * H, generator=g).to(DEV)
    floats = ops.scan_state_floats("matrix_memory" if kind == "memory" else "delta_rule", H, dk, dv)
    state = torch.zeros(4, floats, device=DEV)
    state[:, :] = torch.rand(4, 1, generator=g).to(DEV) * 0.1
    found = []
    for q_lens, slots, run in ((lens, [0, 2, 3][:len(lens)], slice(0, T)), ([mine], [2], slice(at, at + mine))):
        batch = make_batch(q_lens, slots, [0] * len(q_lens), DEV)
        batch.max_q_len = max(q_lens)
        n, st = sum(q_lens), state.clone()
        out = torch.full((n, H * dv), float("nan"), device=DEV)
        x, z = rows[run].clone(), gates[run].clone()
        if kind == "memory":
            ops.matrix_memory_scan(x, 0, H * dk, 2 * H * dk, z, bias, st, batch, H, dk, dv, 15.0, dk ** -0.5, 1e-6, out)
        else:
            ops.delta_rule_scan(x.float(), z, bias[:H].contiguous(), bias[H:].contiguous(), st, batch, H, H, dk, dv, out)
        assert torch.isfinite(out).all()
        found.append((out[at:at + mine] if n == T else out, st[2]))
    assert torch.equal(found[0][0], found[1][0]) and torch.equal(found[0][1], found[1][1])


@pytest.mark.parametrize("kind", ["memory", "delta"])
@pytest.mark.parametrize("mine,least", [(63, 64), (64, 64), (17, 64)])
def test_where_chunks_begin(kind, mine, least):
    """bfloat16 portions below the edge are walked token by token, from it on in chunks: the forced forms' bits."""
    ops = kernels.current()
    H, dk, dv = 2, 64, 24
    g = torch.Generator().manual_seed(mine)
    rows, z = (torch.randn(mine, 2 * H * dk + H * dv, generator=g) * 0.3).to(torch.bfloat16).to(DEV), torch.randn(mine, 2 * H, generator=g).to(DEV)
    bias, found = torch.randn(2 * H, generator=g).to(DEV), []
    for form in (None, mine >= least):
        batch = make_batch([mine], [0], [1], DEV)
        batch.max_q_len = mine
        out, st = torch.empty(mine, H * dv, device=DEV), torch.zeros(1, ops.scan_state_floats("matrix_memory", H, dk, dv), device=DEV)
        if kind == "memory":
            ops.matrix_memory_scan(rows, 0, H * dk, 2 * H * dk, z, bias, st, batch, H, dk, dv, 15.0, dk ** -0.5, 1e-6, out, chunks=form)
        else:
            ops.delta_rule_scan(rows.float(), z.clone(), bias[:H].contiguous(), bias[H:].contiguous(), st, batch, H, H, dk, dv, out,
                                chunks=form)
        found.append(out)
    assert torch.equal(found[0], found[1])
