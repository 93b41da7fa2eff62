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


@pytest.mark.parametrize("n_streams,events", [(0, False), (3, False), (0, True), (2, True)])
@pytest.mark.parametrize("sizes", [[], [7], [0, 3], [800, 700, 900], [1, 0, 2100, 30, 4]], ids=str)
def test_launches_hold_their_requests_by_destination_id(moved, sizes, n_streams, events):
    """Uploaded ids: one launch per request with events, one per stream without, each
    holding its own requests' pairs in ascending destination order."""
    tables = requests(sizes, np.array) if sizes else []
    evs = [SimpleNamespace(cuda_event=1) for _ in sizes] if events else None
    got = moved(tables, n_streams, evs)
    step = len(sizes) if events else max(n_streams, 1)
    want = [sorted(pairs(tables[k::step]), key=lambda p: p[1])
            for k in range(min(step, len(sizes)))]
    assert [g for g in got if g] == [w for w in want if w]


@pytest.mark.parametrize("sizes", [[1500, 1500], [2049], [1000, 1000, 1000]], ids=str)
def test_ids_of_lists_over_the_merge_limit_are_not_read_twice(sizes):
    """Whether lists are merged is decided by their lengths: no id is read for arrays that
    are then thrown away."""
    reads = []

    class Id:
        def __index__(self):
            reads.append(1)
            return 0

    assert copier_module._merged_tables([([Id()] * n, [Id()] * n) for n in sizes]) is None
    assert not reads


@pytest.mark.parametrize("bad,error", [
    (([1, 2], [3, 3]), ValueError), (([1, 2], [3, BLOCKS]), IndexError),
    (([-1, 2], [3, 4]), IndexError), (([1, 2], [2**31, 4]), IndexError),
    (([2**40, 2], [3, 4]), IndexError), (([1, 2], [-2**31, 4]), IndexError)], ids=str)
def test_uploaded_ids_are_refused_before_anything_is_enqueued(moved, bad, error):
    pool = Pool(num_blocks=BLOCKS, native=SimpleNamespace(handle=None))
    for n_streams in (0, 2):
        with pytest.raises(error):
            moved(requests([4, 4], np.array) + [tuple(map(np.array, bad))], n_streams)
    with pytest.raises(ValueError, match="disjoint"):
        moved([(np.array([1]), np.array([2])), (np.array([2]), np.array([3]))], 2,
              pools=(pool, pool))


def test_ordering_long_requests_costs_no_more_than_an_argsort_of_each():
    """Host time of the ids of 64 requests of 256 pairs, on one stream and on two: one
    sort of keys per launch against an argsort per request and a sort for repeats (which
    an earlier lexsort over all pairs exceeded by half)."""
    import time

    pool = Pool(num_blocks=BLOCKS)
    tables = requests([256] * 64, np.array)

    def each():
        src, dst = [], []
        for s, d in tables:
            order = np.argsort(d, kind="stable")
            src.append(s[order])
            dst.append(d[order])
        return pool.host_ids(np.concatenate(src)), pool.host_ids(np.concatenate(dst), unique=True)

    def seconds(work):
        start = time.perf_counter()
        work()
        return time.perf_counter() - start

    for counts in ([64 * 256], [32 * 256] * 2):
        order = lambda: copier_module._launch_order(pool, pool, tables, counts)  # noqa: E731
        times = [(seconds(order), seconds(each)) for _ in range(9)]
        assert min(t[0] for t in times) < min(t[1] for t in times)
