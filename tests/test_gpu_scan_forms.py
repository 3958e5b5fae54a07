"""Which form a recurrence takes, token by token or in chunks: what may depend on it and what may not."""
import json
import os

import pytest
import torch

from helpers import random_tokens, run_plan
from kobolix_helpers import _attn, _delta, _dense, _memory, draw_weights
from reinfer_amd.engine import ModelRunner
from reinfer_amd.weights.safetensors_io import write_safetensors

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
