import os
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
for p in (ROOT, HERE):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (run with -m gpu on the GPU box)")


def pytest_collection_modifyitems(config, items):
    import torch
    if torch.cuda.is_available():
        return
    skip = pytest.mark.skip(reason="no GPU here")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)


@pytest.fixture
def library_calls(monkeypatch):
    """``library_calls(run)``: the names of the kernel library's calls that ``run()`` makes."""
    from reinfer_amd.kernels import library

    def of(run):
        names, call = [], library.call
        with monkeypatch.context() as m:
            m.setattr(library, "call", lambda name, *args: (names.append(name), call(name, *args))[1])
            run()
        return names
    return of
