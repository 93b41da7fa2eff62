"""``HipSlotCopier.copy_requests`` up to the library call, on the CPU.

The copier here is the real method over pools that only know their sizes; streams,
events and the id upload are stand-ins, and the library's entry points record what they
are handed. No kernel runs, so what is checked is which pairs are moved, in which
launches, and what preparing them costs the host.
"""
import ctypes
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from iekv.engine import copier as copier_module
from iekv.engine.copier import HipSlotCopier
from iekv.engine.pools import KVPool

BLOCKS = 40_000


class Pool(SimpleNamespace):
    """The parts of a KVPool the id preparation uses."""

    host_ids = KVPool.host_ids

    def same_shape(self, other):
        return True

    def same_pool_as(self, other):
        return other is self


class Stream(SimpleNamespace):
    def wait_stream(self, other):
        pass

    def wait_event(self, event):
        pass


def stand_in(pool):
    return SimpleNamespace(pool=pool, device="gpu", blocks_read=0, blocks_written=0,
                           flush=lambda: None)


@pytest.fixture
def moved(monkeypatch):
    """copy_requests with the library replaced: call(tables, ...) returns the launches it
    asked for, each a list of (source, destination) pairs, in the order given."""
    current = Stream(device="gpu", cuda_stream=1)
    launches = []

    def library(name, src, dst, *args):
        if name == "iekv_copy_direct_ids":
            s, d, n, _ = args
            s, d = (np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_int32)), (n,))
                    if n else np.empty(0, np.int32) for p in (s, d))
            launches.append(list(zip(s.tolist(), d.tolist())))
            return
        assert name == "iekv_copy_direct_requests"
        k, counts, s, d = args[:4]
        counts = np.ctypeslib.as_array(ctypes.cast(counts, ctypes.POINTER(ctypes.c_int32)), (k,))
        n = int(counts.sum())
        s, d = (np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_int32)), (n,)).tolist()
                if n else [] for p in (s, d))
        at = 0
        for c in counts:
            launches.append(list(zip(s[at:at + c], d[at:at + c])))
            at += c

    monkeypatch.setattr(copier_module._native, "call", library)
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda self, stream: None)
    monkeypatch.setattr(copier_module, "stage_ids", lambda device, *arrays: [
        torch.from_numpy(a.astype(np.int32)) for a in arrays])
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: current)
    monkeypatch.setattr(torch.cuda, "Event", lambda: SimpleNamespace(
        record=lambda s: None, cuda_event=1))
    handle = SimpleNamespace(handle=None)

    def call(tables, n_streams=0, events=None, pools=None):
        src, dst = pools or (Pool(num_blocks=BLOCKS, native=handle),
                             Pool(num_blocks=BLOCKS, native=handle))
        source, dest = stand_in(src), stand_in(dst)
        del launches[:]
        streams = [Stream(device="gpu", cuda_stream=2 + i) for i in range(n_streams)] or None
        HipSlotCopier.copy_requests(dest, source, tables, streams=streams, done_events=events)
        assert source.blocks_read == dest.blocks_written == sum(map(len, launches))
        return [list(x) for x in launches]

    return call


def requests(sizes, form=list, seed=0):
    rng = np.random.default_rng(seed)
    n = sum(sizes)
    src, dst = rng.permutation(BLOCKS)[:n], rng.permutation(BLOCKS)[:n]
    cuts = np.cumsum(sizes)[:-1]
    return [(form(s.tolist()), form(d.tolist()))
            for s, d in zip(np.split(src, cuts), np.split(dst, cuts))]


def pairs(tables):
    return sorted((int(s), int(d)) for src, dst in tables for s, d in zip(src, dst))


@pytest.mark.parametrize("form", [list, tuple, np.array], ids=["list", "tuple", "numpy"])
@pytest.mark.parametrize("n_streams", [0, 2])
@pytest.mark.parametrize("sizes", [[3, 4], [1500, 1500], [2048], [2049], [2, 0, 5, 2100]], ids=str)
def test_tables_given_as_an_iterator_all_move(moved, sizes, n_streams, form):
    """Requests that come from zip(), map() or a generator are read once: whichever way
    their ids take, every request's pairs reach the library."""
    tables = requests(sizes, form)
    want = pairs(tables)
    given = zip([t[0] for t in tables], [t[1] for t in tables])
    assert sorted(sum(moved(given, n_streams), [])) == want
    assert sorted(sum(moved((t for t in tables), n_streams), [])) == want
