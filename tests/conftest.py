import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a HIP GPU (MI355X) and libglif.so")


def gpu_available():
    try:
        import torch
        return torch.cuda.is_available()
    except Exception:
        return False


def pytest_collection_modifyitems(config, items):
    if gpu_available():
        return
    skip = pytest.mark.skip(reason="no GPU visible")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)


@pytest.fixture(params=["windows", "per_tick"])
def both_forwards(request, monkeypatch):
    """The test twice: its cells' forward by windows of three ticks (where the network allows them), and by a
    launch per tick."""
    from v1_glif_model_amd import models
    init = models.V1Column.__init__

    def with_form(self, *args, **kw):
        init(self, *args, **kw)
        self.set_forward(per_tick=request.param == "per_tick")
    monkeypatch.setattr(models.V1Column, "__init__", with_form)
    return request.param
