"""Slot scatter (write_kv) and paged gather (gather_context) kernels vs the NumPy oracle (GPU)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle.slots import gather_context, write_kv

pytestmark = pytest.mark.gpu

CASES = [  # block_size, heads, dim, dtype
    (16, 8, 128, torch.bfloat16),
    (16, 2, 16, torch.float32),
    (4, 1, 2, torch.float32),
    (3, 1, 5, torch.float16),     # 10-byte rows: 2-byte vectors
    (16, 8, 128, torch.float8_e4m3fn),
    (5, 3, 3, torch.uint8),       # 9-byte rows
    (4, 16, 128, torch.float32),  # 8 KiB rows: two steps of four vectors per lane
    (2, 9, 128, torch.float32),   # 4.5 KiB rows: a full step, then 32 lanes
]


def as_np(t: torch.Tensor) -> np.ndarray:
    return t.contiguous().view(torch.uint8).cpu().numpy().copy()


def random_pool(num_blocks, bs, heads, dim, dtype, device, layers=2, seed=0):
    from iekv.engine.pools import KVPool, allocate_pool

    k, v = allocate_pool(num_blocks, bs, layers, heads, dim, dtype=dtype, device=device,
                         zero=False)
    k[0]._base.view(torch.uint8).random_(0, 256,
                                          generator=torch.Generator(device).manual_seed(seed))
    return k, v, KVPool(k, v, bs)


def random_rows(n, heads, dim, dtype, device, seed):
    raw = torch.randint(0, 256, (n, heads, dim * torch.tensor([], dtype=dtype).element_size()),
                        dtype=torch.uint8, device=device,
                        generator=torch.Generator(device).manual_seed(seed))
    return raw.view(dtype)


@pytest.mark.parametrize("bs,heads,dim,dtype", CASES)
def test_write_slots_matches_write_kv(gpu, bs, heads, dim, dtype):
    from iekv.engine.slots import write_slots

    k, v, pool = random_pool(20, bs, heads, dim, dtype, gpu, seed=1)
    oracle_k = [as_np(t) for t in k]
    oracle_v = [as_np(t) for t in v]
    rng = np.random.default_rng(2)
    slots = [int(s) for s in rng.permutation(20 * bs)[:13]]
    for layer in range(2):
        kr = random_rows(13, heads, dim, dtype, gpu, seed=10 + layer)
        vr = random_rows(13, heads, dim, dtype, gpu, seed=20 + layer)
        write_slots(pool, layer, kr, vr, slots)
        write_kv(as_np(kr), as_np(vr), oracle_k[layer], oracle_v[layer], slots)
    torch.cuda.synchronize()
    for got, want in zip(k + v, oracle_k + oracle_v):
        assert np.array_equal(as_np(got), want)


@pytest.mark.parametrize("bs,heads,dim,dtype", CASES)
def test_gather_rows_matches_gather_context(gpu, bs, heads, dim, dtype):
    from iekv.engine.slots import gather_rows

    k, v, pool = random_pool(20, bs, heads, dim, dtype, gpu, seed=3)
    rng = np.random.default_rng(4)
    for context_len in (1, bs, 3 * bs + 1, 7 * bs):
        needed = -(-context_len // bs)
        table = [int(b) for b in rng.permutation(20)[:needed]] + [-1, -1]  # padded like layouts
        for array, cache in enumerate(k + v):
            got = gather_rows(pool, array, table, context_len)
            want = gather_context(as_np(cache), table, context_len, bs)
            assert np.array_equal(as_np(got), want), (context_len, array)


@pytest.mark.parametrize("bs,heads,dim,dtype", CASES)
def test_one_launch_writes_every_layer_like_write_kv_per_layer(gpu, bs, heads, dim, dtype):
    """iekv_write_slots_layers: all four layers at once, then layers 1..2 with new
    rows, then (layer_stride 0) the same rows into every layer; each against the
    oracle's write_kv per layer."""
    from iekv import _native
    from iekv.engine.slots import write_slots_layers

    L = 4
    k, v, pool = random_pool(20, bs, heads, dim, dtype, gpu, layers=L, seed=5)
    oracle_k = [as_np(t) for t in k]
    oracle_v = [as_np(t) for t in v]
    rng = np.random.default_rng(6)
    for first, n_layers, seed in ((0, L, 30), (1, 2, 40)):
        slots = [int(x) for x in rng.permutation(20 * bs)[:13]]
        kr = random_rows(n_layers * 13, heads, dim, dtype, gpu, seed).view(n_layers, 13, heads, dim)
        vr = random_rows(n_layers * 13, heads, dim, dtype, gpu, seed + 1).view(
            n_layers, 13, heads, dim)
        write_slots_layers(pool, kr, vr, slots, first_layer=first)
        for l in range(n_layers):
            write_kv(as_np(kr[l]), as_np(vr[l]), oracle_k[first + l], oracle_v[first + l], slots)
    slots = [int(x) for x in rng.permutation(20 * bs)[:7]]
    kr, vr = (random_rows(7, heads, dim, dtype, gpu, seed) for seed in (50, 51))
    dev_slots = torch.tensor(slots, dtype=torch.int64, device=gpu)
    _native.call("iekv_write_slots_layers", pool.native.handle, 0, L, bs, kr.data_ptr(),
                 vr.data_ptr(), 0, dev_slots.data_ptr(), 7,
                 torch.cuda.current_stream().cuda_stream)
    for l in range(L):
        write_kv(as_np(kr), as_np(vr), oracle_k[l], oracle_v[l], slots)
    torch.cuda.synchronize()
    for got, want in zip(k + v, oracle_k + oracle_v):
        assert np.array_equal(as_np(got), want)


@pytest.mark.parametrize("bs,heads,dim,dtype", CASES)
def test_one_launch_gathers_every_array_like_gather_context(gpu, bs, heads, dim, dtype):
    from iekv.engine.slots import gather_rows_arrays

    k, v, pool = random_pool(20, bs, heads, dim, dtype, gpu, layers=3, seed=7)
    rng = np.random.default_rng(8)
    for context_len in (1, bs, 3 * bs + 1, 7 * bs):
        needed = -(-context_len // bs)
        table = [int(b) for b in rng.permutation(20)[:needed]] + [-1]
        got = gather_rows_arrays(pool, table, context_len)
        assert got.shape[:2] == (6, context_len)
        for array, cache in enumerate(k + v):
            want = gather_context(as_np(cache), table, context_len, bs)
            assert np.array_equal(as_np(got[array]), want), (context_len, array)
        part = gather_rows_arrays(pool, table, context_len, first_array=2, n_arrays=3)
        assert torch.equal(part.view(torch.uint8), got[2:5].contiguous().view(torch.uint8))


def test_slot_calls_validate_before_launch(gpu):
    from iekv.engine.slots import gather_rows, write_slots

    k, v, pool = random_pool(4, 4, 1, 2, torch.float32, gpu)
    rows = torch.zeros(2, 1, 2, device=gpu)
    with pytest.raises(IndexError):
        write_slots(pool, 0, rows, rows, [0, 16])
    with pytest.raises(IndexError):
        write_slots(pool, 2, rows, rows, [0, 1])
    with pytest.raises(ValueError):
        write_slots(pool, 0, rows, rows, [0])
    with pytest.raises(IndexError):
        gather_rows(pool, 0, [3], 6)
    from iekv.engine.slots import gather_rows_arrays, write_slots_layers

    with pytest.raises(IndexError):
        write_slots_layers(pool, rows[None].expand(2, -1, -1, -1), rows[None].expand(2, -1, -1, -1),
                           [0, 1], first_layer=1)
    with pytest.raises(IndexError):
        gather_rows_arrays(pool, [0, 1], 6, first_array=3, n_arrays=2)


@pytest.mark.parametrize("cache_dtype", [torch.float32, torch.bfloat16], ids=str)
def test_the_model_decodes_identically_through_the_slot_kernels(gpu, cache_dtype):
    from conftest import golden
    from iekv.engine.engine import Engine, EngineConfig
    from iekv.engine.toy_model import ModelConfig, ToyTransformer
    from iekv.serve.disaggregated import DisaggregatedEngine

    g = golden("disaggregation")
    cfg = EngineConfig(**g["engine"])

    def model(hip_kv):
        return ToyTransformer(ModelConfig(**g["model"]), seed=g["model_seed"], device=gpu,
                              cache_dtype=cache_dtype, hip_kv=hip_kv)

    torch_path = Engine(model(False), cfg).generate(g["prompts"], max_new_tokens=6,
                                                    temperature=0.0)
    hip_colocated = Engine(model(True), cfg).generate(g["prompts"], max_new_tokens=6,
                                                      temperature=0.0)
    hip_split = DisaggregatedEngine(model(True), cfg, mode="direct").generate(
        g["prompts"], max_new_tokens=6, temperature=0.0)
    assert hip_colocated == torch_path == hip_split


def test_slots_and_table_entries_at_the_top_of_a_pool_of_int32_max_blocks(gpu):
    """A pool of INT32_MAX blocks of 2 slots (8-byte rows, one layer's K and V: 64 GiB)
    has 2^32 - 2 slots: write_kv's int64 slots above 2^32 - 5 and past 2^31, and
    gather_context's table entries next to INT32_MAX, address rows 32 GiB into each
    array. Both kernels move exactly those rows, and the rows beside each written one
    keep their bytes."""
    from iekv.engine.pools import KVPool, allocate_pool
    from iekv.engine.slots import gather_rows_arrays, write_slots_layers

    n, bs = 2**31 - 1, 2
    rows = n * bs
    k, v = allocate_pool(n, bs, 1, 1, 8, dtype=torch.uint8, device=gpu, zero=False)
    pool = KVPool(k, v, bs)
    gen = torch.Generator(gpu).manual_seed(71)
    slots = [rows - 1, rows - 4, 5, 2**31 + 7, 2**32 - 9]
    beside = sorted({s + d for s in slots for d in (-1, 1) if 0 <= s + d < rows} - set(slots))
    idx = torch.tensor(beside, dtype=torch.long, device=gpu)
    for arr in (k[0], v[0]):
        arr.view(rows, 8).index_copy_(0, idx, torch.randint(
            0, 256, (len(beside), 8), dtype=torch.uint8, device=gpu, generator=gen))
    kept = [arr.view(rows, 8)[idx].clone() for arr in (k[0], v[0])]
    new_k = torch.randint(0, 256, (1, len(slots), 1, 8), dtype=torch.uint8, device=gpu,
                          generator=gen)
    new_v = torch.randint(0, 256, (1, len(slots), 1, 8), dtype=torch.uint8, device=gpu,
                          generator=gen)
    print("int32-limit slot pool: write_kv", flush=True)
    write_slots_layers(pool, new_k, new_v, slots)
    torch.cuda.synchronize()
    sl = torch.tensor(slots, dtype=torch.long, device=gpu)
    assert torch.equal(k[0].view(rows, 8)[sl], new_k[0].view(-1, 8))
    assert torch.equal(v[0].view(rows, 8)[sl], new_v[0].view(-1, 8))
    for arr, before in zip((k[0], v[0]), kept):
        assert torch.equal(arr.view(rows, 8)[idx], before)
    # gather_context over a table whose blocks sit at the top of the pool
    table = [n - 1, n - 2, 3, n - 5]
    context = 7                                          # the last block half used
    want_rows = torch.tensor([table[j // bs] * bs + j % bs for j in range(context)],
                             dtype=torch.long, device=gpu)
    for arr in (k[0], v[0]):
        arr.view(rows, 8).index_copy_(0, want_rows, torch.randint(
            0, 256, (context, 8), dtype=torch.uint8, device=gpu, generator=gen))
    print("int32-limit slot pool: gather_context", flush=True)
    out = gather_rows_arrays(pool, table, context)
    torch.cuda.synchronize()
    for a, arr in enumerate((k[0], v[0])):
        assert torch.equal(out[a].view(context, 8), arr.view(rows, 8)[want_rows])
    pool.native.close()
    del k, v, pool, out
    torch.cuda.empty_cache()


def test_gather_takes_the_block_table_as_a_list_or_a_tensor(gpu):
    """A decode loop may keep its block tables on the GPU or in a CPU tensor:
    gather_context and the every-array gather read the same rows through a device
    int32 or int64 tensor, a CPU tensor and a Python list, and a table too short
    for the context raises IndexError in every form, as the reference's does."""
    from iekv.engine.slots import gather_rows, gather_rows_arrays

    bs, heads, dim = 4, 2, 16
    k, v, pool = random_pool(30, bs, heads, dim, torch.float16, gpu, seed=91)
    table, context = [17, 2, 29, 8], 14
    raw = lambda t: t.view(torch.uint8)       # NaN bit patterns compare as bytes
    want = gather_rows_arrays(pool, table, context)
    for form in (torch.tensor(table, dtype=torch.int32, device=gpu),
                 torch.tensor(table, dtype=torch.int64, device=gpu),
                 torch.tensor(table, dtype=torch.int32)):
        assert torch.equal(raw(gather_rows_arrays(pool, form, context)), raw(want))
        for array in (0, 3):
            assert torch.equal(raw(gather_rows(pool, array, form, context)), raw(want[array]))
        with pytest.raises(IndexError):
            gather_rows_arrays(pool, form[:3], context)
        with pytest.raises(IndexError):
            gather_rows(pool, 0, form[:3], context)
    oracle = gather_context(as_np(k[1]), table, context, bs)
    assert np.array_equal(as_np(want[1]), oracle.reshape(as_np(want[1]).shape))


@pytest.mark.parametrize("bs,heads,dim,dtype", [
    (2, 8, 128, torch.bfloat16),   # 256 vectors per block: one workgroup each
    (1, 5, 80, torch.float16),     # 50 vectors per block: workgroups span blocks
    (3, 1, 5, torch.float16),      # 30-byte blocks: the width follows the context's length
])
@pytest.mark.parametrize("blocks", [1, 64, 65, 512, 513, 1030])
def test_host_tables_gather_like_device_tables_around_the_launch_limits(gpu, bs, heads, dim,
                                                                        dtype, blocks):
    """A list table rides in the launch's arguments (64 or 512 entries, longer ones in
    several launches), a device table stays where it is: both read the rows the oracle
    reads, with whole and partial last blocks."""
    from iekv.engine.slots import gather_rows_arrays

    n = 1040
    k, v, pool = random_pool(n, bs, heads, dim, dtype, gpu, layers=2, seed=101)
    table = [int(b) for b in np.random.default_rng(blocks).permutation(n)[:blocks]]
    on_device = torch.tensor(table, dtype=torch.int32, device=gpu)
    caches = [as_np(c) for c in k + v]
    for context in {blocks * bs, (blocks - 1) * bs + 1}:
        got = gather_rows_arrays(pool, table, context)
        want = gather_rows_arrays(pool, on_device, context)
        assert torch.equal(got.view(torch.uint8), want.view(torch.uint8))
        for a, cache in enumerate(caches):
            oracle = gather_context(cache, table, context, bs)
            assert np.array_equal(as_np(got[a]).reshape(oracle.shape), oracle), (a, context)
    for bad in (-1, n):
        with pytest.raises(IndexError, match="context block id"):
            gather_rows_arrays(pool, table[:-1] + [bad], blocks * bs)
    with pytest.raises(TypeError):
        gather_rows_arrays(pool, table[:-1] + [1.5], blocks * bs)


@pytest.mark.parametrize("bs,heads,dim", [
    (4, 8, 128),    # 1,024-element rows: 16-byte vectors
    (2, 5, 80),     # rows of 100 and 25 source vectors: workgroups span rows
    (3, 1, 6),      # rows that hold no whole 16-byte vector: one element per lane
])
@pytest.mark.parametrize("row_dtype,cache_dtype", [
    (torch.float32, torch.float16), (torch.float32, torch.bfloat16),
    (torch.float32, torch.float8_e4m3fn), (torch.float16, torch.float8_e4m3fn),
    (torch.bfloat16, torch.float8_e4m3fn), (torch.float16, torch.float16),
    (torch.float16, torch.float32),          # a pair torch casts first
], ids=str)
def test_rows_of_another_type_are_written_as_their_casts(gpu, bs, heads, dim, row_dtype,
                                                         cache_dtype):
    """Rows rounded on their way to the cache equal index_copy_ of k.to(cache dtype), NaNs,
    infinities, overflows, ties and denormals included; slots as a list that one launch's
    arguments hold, one that takes a longer block or two launches, one that is uploaded,
    and a device tensor; aligned and odd row addresses."""
    from iekv.engine.slots import write_slots, write_slots_layers

    n_blocks = 700 // bs
    rows_in_pool = n_blocks * bs
    special = torch.tensor([0.0, -0.0, 1e-45, -3e-8, 6e-5, 447.9, 448.0, 456.0, 464.0, 464.1,
                            480.0, -500.0, 65504.0, 65520.0, 1e30, float("inf"), -float("inf"),
                            float("nan"), -float("nan"), 1.00390625, 0.0625 * 1.0625])
    for n in (1, 64, 65, 256, 257, 512, 513):
        k, v, pool = random_pool(n_blocks, bs, heads, dim, cache_dtype, gpu, layers=3, seed=n)
        want = [c.clone() for c in k + v]
        gen = torch.Generator(gpu).manual_seed(200 + n)
        total = 2 * 2 * n * heads * dim
        flat = torch.randn(total + 1, device=gpu, generator=gen) * 100
        at = torch.randint(0, total, (total // 4 + 1,), device=gpu, generator=gen)
        flat[at] = special.to(gpu)[torch.randint(0, special.numel(), at.shape, device=gpu,
                                                 generator=gen)]
        odd = n % 2                                 # odd: rows start one element in
        rows = flat.to(row_dtype)[odd:odd + total].view(2, 2, n, heads, dim)
        slots = [int(s) for s in np.random.default_rng(n).permutation(rows_in_pool)[:n]]
        where = torch.tensor(slots, device=gpu)
        write_slots_layers(pool, rows[0], rows[1], slots if n != 65 else where, first_layer=1)
        for l in range(2):
            want[1 + l].view(torch.uint8)[where] = rows[0, l].to(cache_dtype).view(torch.uint8)
            want[4 + l].view(torch.uint8)[where] = rows[1, l].to(cache_dtype).view(torch.uint8)
        write_slots(pool, 0, rows[1, 0], rows[0, 1], where if n != 65 else slots)
        want[0].view(torch.uint8)[where] = rows[1, 0].to(cache_dtype).view(torch.uint8)
        want[3].view(torch.uint8)[where] = rows[0, 1].to(cache_dtype).view(torch.uint8)
        for a, (got, expected) in enumerate(zip(k + v, want)):
            assert torch.equal(got.view(torch.uint8), expected.view(torch.uint8)), (n, a)
        for bad in (-1, rows_in_pool):
            with pytest.raises(IndexError, match=f"slot {bad} out of range"):
                write_slots_layers(pool, rows[0], rows[1], slots[:-1] + [bad])


def test_captured_writes_replay_and_uploads_are_refused_under_capture(gpu):
    """A list that rides in the launches' arguments and a device tensor are captured and
    write the rows' present values on every replay; a longer list, which is uploaded from
    memory that does not outlive the call, is refused and leaves the capture whole."""
    from iekv.engine.slots import HOST_SLOTS_MAX, write_slots

    k, v, pool = random_pool(70, 16, 2, 32, torch.float16, gpu, layers=1, seed=5)
    n = HOST_SLOTS_MAX
    order = np.random.default_rng(6).permutation(70 * 16)
    slots, tensor = order[:n].tolist(), torch.from_numpy(order[n:2 * n].copy()).to(gpu)
    rows = torch.zeros((n + 1, 2, 32), dtype=torch.float32, device=gpu)
    write_slots(pool, 0, rows[:n], rows[:n], slots)      # first use outside the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        with pytest.raises(RuntimeError, match="under capture"):
            write_slots(pool, 0, rows, rows, order[:n + 1].tolist())
        write_slots(pool, 0, rows[:n], rows[:n], slots)
        write_slots(pool, 0, rows[:n], rows[:n], tensor)
    for step in range(4):
        rows.copy_(torch.randn(rows.shape, device=gpu,
                               generator=torch.Generator(gpu).manual_seed(step)))
        want = [c.clone() for c in k + v]
        for w in want:
            w[torch.tensor(slots, device=gpu)] = rows[:n].half()
            w[tensor] = rows[:n].half()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(w.view(torch.int16), c.view(torch.int16))
                   for w, c in zip(want, k + v)), step      # bytes: the pool holds NaNs


@pytest.mark.parametrize("row", [1, 2, 7, 8, 12, 15, 16, 17, 24, 31, 33, 162, 1000, 2056])
@pytest.mark.parametrize("offset", [0, 1, 2, 4, 8])
def test_rows_of_any_size_at_any_address_are_written(gpu, row, offset):
    """Rows of bytes on either side of one 16-byte vector, whole ones and not, at addresses
    that are multiples of 16, 8, 4, 2 and 1: every row lands in its slot, the bytes of the
    other slots stay, and so do those beside the arrays."""
    from iekv.engine.pools import KVPool, allocate_pool
    from iekv.engine.slots import write_slots_layers

    for n in (1, 16, 257, 600):
        k, v = allocate_pool(41, 16, 2, 1, row, dtype=torch.uint8, device=gpu, zero=False,
                             pad_blocks=1)
        slab = k[0]._base
        slab.random_(0, 256, generator=torch.Generator(gpu).manual_seed(n))
        pool = KVPool(k, v, 16)
        total = 2 * n * row
        flat = torch.randint(0, 256, (2 * total + 32,), dtype=torch.uint8, device=gpu,
                             generator=torch.Generator(gpu).manual_seed(row))
        rows_k = flat[offset:offset + total].view(2, n, 1, row)
        rows_v = flat[total + 16:2 * total + 16].view(2, n, 1, row)
        where = torch.from_numpy(np.random.default_rng(n + row).permutation(41 * 16)[:n]).to(gpu)
        want = slab.clone()
        for l in range(2):
            want[0, l, where] = rows_k[l]
            want[1, l, where] = rows_v[l]
        write_slots_layers(pool, rows_k, rows_v, where if n != 257 else where.tolist())
        assert torch.equal(slab, want), n


@pytest.mark.parametrize("elems", [3, 4, 5, 7, 8, 9, 15, 27, 125, 256])
@pytest.mark.parametrize("row_dtype,cache_dtype", [
    (torch.float32, torch.float16), (torch.float32, torch.bfloat16),
    (torch.float32, torch.float8_e4m3fn), (torch.float16, torch.float8_e4m3fn),
    (torch.bfloat16, torch.float8_e4m3fn)], ids=str)
def test_casts_of_any_row_size_at_any_address(gpu, elems, row_dtype, cache_dtype):
    """Rows of another type on either side of one vector's elements, whole vectors and not,
    aligned and one element in, with one launch and several (host lists over 256 slots),
    an upload and device slots: each equals torch's cast, and nothing else changes."""
    from iekv.engine.pools import KVPool, allocate_pool
    from iekv.engine.slots import write_slots_layers

    for n in (1, 65, 257, 513):
        for first in (0, 1):
            k, v = allocate_pool(66, 8, 2, 1, elems, dtype=cache_dtype, device=gpu, zero=False,
                                 pad_blocks=1)
            slab = k[0]._base.view(torch.uint8)
            slab.random_(0, 256, generator=torch.Generator(gpu).manual_seed(n))
            pool = KVPool(k, v, 8)
            total = 2 * n * elems
            pad = -total % 16 + 16
            flat = (torch.randn(2 * total + 2 * pad, device=gpu,
                                generator=torch.Generator(gpu).manual_seed(elems)) * 50
                    ).to(row_dtype)
            rows_k = flat[first:first + total].view(2, n, 1, elems)
            rows_v = flat[total + pad:2 * total + pad].view(2, n, 1, elems)
            where = torch.from_numpy(np.random.default_rng(n).permutation(66 * 8)[:n]).to(gpu)
            want = slab.clone()
            for l in range(2):
                want[0, l, where] = rows_k[l].to(cache_dtype).view(torch.uint8)
                want[1, l, where] = rows_v[l].to(cache_dtype).view(torch.uint8)
            write_slots_layers(pool, rows_k, rows_v, where if n == 65 else where.tolist())
            assert torch.equal(slab, want), (n, first)


@pytest.mark.parametrize("row", [1, 3, 7, 8, 12, 15, 16, 17, 24, 31, 162, 1000, 2056])
@pytest.mark.parametrize("offset", [0, 1, 8])
def test_contexts_of_any_row_size_are_gathered_to_any_address(gpu, row, offset):
    """Contexts of blocks on either side of one 16-byte vector, whole ones and not, last
    blocks of one row and of all, into outputs at multiples of 16, 8 and 1 bytes, by host
    and by device tables: every byte of every context, and none beside them."""
    from iekv import _native
    from iekv.engine.pools import KVPool, allocate_pool, current_stream_handle

    for bs in (1, 5, 16):
        k, v = allocate_pool(530, bs, 2, 1, row, dtype=torch.uint8, device=gpu, zero=False)
        k[0]._base.random_(0, 256, generator=torch.Generator(gpu).manual_seed(bs))
        pool = KVPool(k, v, bs)
        table = [int(b) for b in np.random.default_rng(row).permutation(530)]
        on_device = torch.tensor(table, dtype=torch.int32, device=gpu)
        on_host = np.array(table, np.int32)
        rows = (on_device.long()[:, None] * bs + torch.arange(bs, device=gpu)).reshape(-1)
        for tokens in {1, bs, bs + 1, 37 * bs, 514 * bs - bs // 2}:
            want = torch.stack([c[rows[:tokens]] for c in k + v]).view(torch.uint8).reshape(-1)
            for fn, address in (("iekv_gather_rows_arrays", on_device.data_ptr()),
                                ("iekv_gather_rows_arrays_ids", on_host.ctypes.data)):
                out = torch.full((want.numel() + 512,), 0xA5, dtype=torch.uint8, device=gpu)
                _native.call(fn, pool.native.handle, 0, 4, bs, address, tokens,
                             out.data_ptr() + 256 + offset, want.numel(),
                             current_stream_handle(pool.device))
                at = 256 + offset
                assert torch.equal(out[at:at + want.numel()], want), (bs, tokens, fn)
                assert bool((out[:at] == 0xA5).all()) and \
                    bool((out[at + want.numel():] == 0xA5).all()), (bs, tokens, fn)


@pytest.mark.parametrize("n", [2047, 2048, 2049, 3584, 3585])
def test_writes_of_one_and_of_two_vectors_a_lane(gpu, n):
    """Aligned rows of one layer around the launch sizes that take two vectors a lane, rows
    of a power of two of vectors and not."""
    from iekv.engine.slots import write_slots

    for dim in (2048, 2064):        # 128 and 129 vectors a row
        k, v, pool = random_pool(230, 16, 1, dim, torch.uint8, gpu, layers=1, seed=n)
        rows = torch.randint(0, 256, (2, n, 1, dim), dtype=torch.uint8, device=gpu,
                             generator=torch.Generator(gpu).manual_seed(dim))
        where = torch.from_numpy(np.random.default_rng(n).permutation(230 * 16)[:n]).to(gpu)
        want = [c.clone() for c in k + v]
        want[0][where], want[1][where] = rows[0], rows[1]
        write_slots(pool, 0, rows[0], rows[1], where)
        assert all(torch.equal(w, c) for w, c in zip(want, k + v)), dim


@pytest.mark.parametrize("blocks", [2047, 2048, 2049, 5000])
def test_long_host_tables_gather_like_device_tables(gpu, blocks):
    """Tables on either side of the longest that rides in launch arguments, as lists and
    arrays: the rows a device table gives; ids outside the pool are refused either way."""
    from iekv.engine.slots import gather_rows, gather_rows_arrays

    k, v, pool = random_pool(5003, 3, 2, 20, torch.float16, gpu, layers=2, seed=blocks)
    table = np.random.default_rng(blocks).permutation(5003)[:blocks]
    on_device = torch.from_numpy(table.astype(np.int32)).to(gpu)
    for context in (blocks * 3, blocks * 3 - 2):
        want = gather_rows_arrays(pool, on_device, context).view(torch.uint8)
        rows = (on_device.long()[:, None] * 3 + torch.arange(3, device=gpu)).reshape(-1)[:context]
        assert torch.equal(want[0], k[0][rows].view(torch.uint8))
        for form in (table.tolist(), table, tuple(table.tolist())):
            assert torch.equal(gather_rows_arrays(pool, form, context).view(torch.uint8), want)
            assert torch.equal(gather_rows(pool, 3, form, context).view(torch.uint8), want[3])
    for bad in (-1, 5003):
        with pytest.raises(IndexError, match="context block id"):
            gather_rows_arrays(pool, table[:-1].tolist() + [bad], blocks * 3)
    with pytest.raises(TypeError):
        gather_rows_arrays(pool, table[:-1].tolist() + [1.5], blocks * 3)


@pytest.mark.parametrize("row_dtype,cache_dtype", [
    (torch.float32, torch.float16), (torch.float32, torch.bfloat16),
    (torch.float32, torch.float8_e4m3fn), (torch.float16, torch.float8_e4m3fn),
    (torch.bfloat16, torch.float8_e4m3fn)], ids=str)
def test_every_value_is_cast_as_torch_casts_it(gpu, row_dtype, cache_dtype):
    """Every bit pattern of the row type, written as rows: the cache holds the bytes of
    torch's cast on the GPU, ties, subnormals, overflow, infinities and NaNs of every
    payload included. Rows aligned, and (the 16-bit types) one element in, which takes
    the vectors at any address."""
    from iekv.engine.slots import write_slots

    bits = 8 * torch.tensor([], dtype=row_dtype).element_size()
    dim, per_call = 1024, min(1 << 26, 1 << (bits - 1))
    n = per_call // dim
    k, v, pool = random_pool(n, 1, 1, dim, cache_dtype, gpu, layers=1, seed=1)
    where = torch.arange(n, device=gpu)
    whole = torch.int32 if bits == 32 else torch.int16
    patterns = torch.arange(per_call, device=gpu, dtype=torch.int64)
    for first in range(-(1 << (bits - 1)), 1 << (bits - 1), 2 * per_call):
        rows = [(patterns + first + half * per_call).to(whole).view(row_dtype).view(n, 1, dim)
                for half in (0, 1)]
        write_slots(pool, 0, rows[0], rows[1], where)
        for cache, row in zip(k + v, rows):
            assert torch.equal(cache.view(torch.uint8),
                               row.to(cache_dtype).view(torch.uint8)), first
        if bits == 16:
            for r in rows:
                moved = torch.cat([r.reshape(-1)[:1], r.reshape(-1)])[1:].view(n, 1, dim)
                assert moved.data_ptr() % 4
                write_slots(pool, 0, moved, moved, where)
                want = r.to(cache_dtype).view(torch.uint8)
                assert all(torch.equal(c.view(torch.uint8), want) for c in k + v), first


def test_row_kernels_with_ordinary_accesses(gpu):
    """The non-temporal setting off: aligned rows and contexts take ordinary accesses, the
    other kinds go on streaming; the same bytes either way."""
    from iekv import _native
    from iekv.engine.slots import gather_rows_arrays, write_slots_layers

    shape = _native.get_launch()
    _native.set_launch(nontemporal=0)
    try:
        for dim, dtype, rows_dtype in ((128, torch.bfloat16, torch.bfloat16),
                                       (81, torch.bfloat16, torch.bfloat16),
                                       (3, torch.float16, torch.float16),
                                       (128, torch.bfloat16, torch.float32)):
            k, v, pool = random_pool(300, 16, 3, dim, dtype, gpu, layers=2, seed=dim)
            n = 1600
            rows = torch.randn(2, 2, n, 3, dim, device=gpu).to(rows_dtype)
            slots = np.random.default_rng(dim).permutation(300 * 16)[:n].tolist()
            where = torch.tensor(slots, device=gpu)
            want = [c.clone().view(torch.int16) for c in k + v]
            for l in range(2):
                want[l][where] = rows[0, l].to(dtype).view(torch.int16)
                want[2 + l][where] = rows[1, l].to(dtype).view(torch.int16)
            write_slots_layers(pool, rows[0], rows[1], where)
            write_slots_layers(pool, rows[0][:, :70].contiguous(), rows[1][:, :70].contiguous(),
                               slots[:70])
            assert all(torch.equal(w, c.view(torch.int16)) for w, c in zip(want, k + v)), dim
            table = np.random.default_rng(dim + 1).permutation(300)[:90].tolist()
            index = (torch.tensor(table, device=gpu)[:, None] * 16 +
                     torch.arange(16, device=gpu)).reshape(-1)[:1437]
            for form in (table, torch.tensor(table, dtype=torch.int32, device=gpu)):
                got = gather_rows_arrays(pool, form, 1437).view(torch.int16)
                assert all(torch.equal(g, w[index]) for g, w in zip(got, want)), dim
    finally:
        _native.set_launch(nontemporal=shape["nontemporal"])
