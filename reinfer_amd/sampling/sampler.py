"""Sampling on the GPU from the step's float32 logits.

Greedy takes the first maximum. Temperature > 0 draws by Gumbel-max with noise
that is a pure function of (request seed, position, token id), so equal logits
give a request the same tokens whatever else is in the batch, however its prompt
was cut and whether or not it was preempted and recomputed (that the logits are
equal to the last bit is a matter of the kernels that the steps went through)
(crates/scheduler/src/rng.rs:52-66; crates/cuda/kernels/sampler_kernel.cu:61-77).
Filters and penalties, if asked for, mask or shift the logits first, in the
reference's order: repeat, frequency/presence, top-k, top-p, min-p, then
temperature and the draw (crates/samplers/src/lib.rs:66-90).
"""
from __future__ import annotations

from typing import List, Optional, Sequence

import numpy as np
import torch

from .. import kernels
from ..kernels.upload import to_device
from .params import SamplingParams

_MASK63 = (1 << 63) - 1


class SamplingError(RuntimeError):
    """No token could be drawn: every logit of a row is non-finite
    (bin/reinfer/src/pipeline.rs:189-191 raises on all-NaN logits)."""


def derive_seed(engine_seed: int, arrival: int) -> int:
    """Seed of a request that brings none: splitmix64(engine seed ^ arrival number)
    (bin/reinfer/src/sched_loop.rs:651-653)."""
    from ..weights.random_init import splitmix64
    return splitmix64((engine_seed ^ arrival) & ((1 << 64) - 1))


def as_int64(seed: int) -> int:
    seed &= (1 << 64) - 1
    return seed - (1 << 64) if seed >= (1 << 63) else seed


class Sampler:
    def __init__(self, device: torch.device):
        self.device = device

    def sample(self, logits: torch.Tensor, params: Sequence[SamplingParams], seeds: Sequence[int],
               positions: Sequence[int], histories: Optional[Sequence[Sequence[int]]] = None) -> List[int]:
        """One token per row of ``logits``; ``positions[i]`` is the index the new
        token will have in its request, ``histories[i]`` the request's tokens so far."""
        n = logits.shape[0]
        if not (len(params) == len(seeds) == len(positions) == n):
            raise ValueError("one SamplingParams, seed and position per row")
        ops = kernels.current()
        if any(p.filters for p in params):
            if histories is None:
                raise ValueError("penalties need the requests' tokens")
            if hasattr(ops, "sample_filtered") and len(histories) == n:
                if logits.stride(1) != 1 or logits.stride(0) < logits.shape[1]:
                    logits = logits.clone()
                tokens = torch.empty(n, dtype=torch.int32, device=self.device)
                ops.sample_filtered(logits, params, histories, [as_int64(int(s)) for s in seeds], [int(p) for p in positions], tokens)
                return self._drawn(tokens)
            # a kernel set without that, or fewer histories than rows (the others' options are not applied)
            logits = logits.clone()
            ops.filter_logits(logits, params, histories)
        # one transfer: seeds, temperatures, positions
        rows = np.empty(16 * n, dtype=np.uint8)
        rows[:8 * n].view(np.int64)[:] = [as_int64(int(s)) for s in seeds]
        rows[8 * n:12 * n].view(np.float32)[:] = [max(0.0, float(p.temperature)) for p in params]
        rows[12 * n:].view(np.int32)[:] = [int(p) for p in positions]
        rows_t = to_device(rows, self.device)
        tokens = torch.empty(n, dtype=torch.int32, device=self.device)
        ops.sample(logits, rows_t[8 * n:12 * n].view(torch.float32), rows_t[:8 * n].view(torch.int64),
                   rows_t[12 * n:].view(torch.int32), tokens)
        return self._drawn(tokens)

    @staticmethod
    def _drawn(tokens: torch.Tensor) -> List[int]:
        out = tokens.tolist()
        for i, t in enumerate(out):
            if t < 0:
                raise SamplingError(f"row {i}: no finite logit to sample from")
        return out
