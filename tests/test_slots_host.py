"""Slot lists of the row writes, checked on the host (no GPU)."""
from contextlib import nullcontext
from types import SimpleNamespace

import pytest
import torch

from iekv.engine import slots as slots_module


def test_a_list_that_would_be_uploaded_is_refused_under_capture(monkeypatch):
    """A replay would read the upload's pinned source again after it was freed; lists that
    ride in the launch's arguments are taken."""
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    monkeypatch.setattr(torch.cuda, "device", lambda device: nullcontext())
    monkeypatch.setattr(torch.Tensor, "pin_memory",
                        lambda self: pytest.fail("uploaded under capture"))
    pool = SimpleNamespace(num_blocks=100, block_size=16, device=torch.device("cuda", 0))
    most = slots_module.HOST_SLOTS_MAX
    with pytest.raises(RuntimeError, match="under capture"):
        slots_module._slots(pool, list(range(most + 1)))
    with pytest.raises(IndexError, match="slot 1600 out of range"):
        slots_module._slots(pool, list(range(most)) + [1600])
    assert slots_module._slots(pool, list(range(most)))[1] == "iekv_write_slots_cast_ids"
