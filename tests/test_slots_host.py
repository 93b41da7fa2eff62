"""Slot lists of the row writes, checked on the host (no GPU)."""
from contextlib import nullcontext
from types import SimpleNamespace

import numpy as np
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


def test_long_tables_are_uploaded_except_under_capture(monkeypatch):
    """Tables of up to HOST_TABLE_MAX blocks ride in the launches' arguments; a longer one is
    checked and uploaded, unless the stream is under capture, where nothing may be."""
    uploads = []
    monkeypatch.setattr(torch.cuda, "device", lambda device: nullcontext())
    pool = SimpleNamespace(block_size=16, device=torch.device("cuda", 0),
                           block_ids=lambda ids, what: uploads.append(len(ids)) or "uploaded")
    most = slots_module.HOST_TABLE_MAX
    for capturing in (False, True):
        monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing)
        for form in (list, tuple, np.array):
            for blocks in (1, 512, most, most + 1, 4 * most):
                del uploads[:]
                table = form(list(range(blocks + 3)))
                ids, fn = slots_module._context_table(pool, table, blocks * 16)
                if blocks > most and not capturing:
                    assert (ids, fn, uploads) == ("uploaded", "iekv_gather_rows_arrays", [blocks])
                else:
                    assert list(ids) == list(range(blocks)) and not uploads
                    assert fn == "iekv_gather_rows_arrays_ids"
