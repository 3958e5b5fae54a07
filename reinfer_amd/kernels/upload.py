"""Small host arrays on their way to a kernel."""
from __future__ import annotations

import numpy as np
import torch


def to_device(array: np.ndarray, device) -> torch.Tensor:
    """``array`` on ``device``. To a GPU from page-locked memory and without waiting (a transfer from ordinary memory ends only
    when it is done: 17 us each at a few KB): the host allocator gives the memory out again once the copy on the current
    stream is over."""
    host = torch.from_numpy(array)
    device = torch.device(device)
    if device.type != "cuda":
        return host.to(device)
    return host.pin_memory().to(device, non_blocking=True)
