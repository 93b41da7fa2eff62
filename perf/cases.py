"""Performance cases of the paged KV-cache handoff, through the package's public entry points.

A case names an operation, a pool geometry and a size. The operations are what a
serving program calls on either side of a prefill -> decode handoff:

  direct    ``HipSlotCopier.copy_blocks`` with block tables as Python lists: one
            finished prefill moves from the prefill pool to the decode pool
  checked   the same with block ids held on the GPU and checked there
            (``check_device_ids=True``)
  requests  ``HipSlotCopier.copy_requests``: several admitted prompts in one call
  transfer  ``read_blocks`` then ``write_blocks``: the handoff through a packed payload
  write     ``write_slots_layers``: one forward step's new K and V rows of every
            layer, scattered by slot (the slots in a list, or a device tensor as a
            model that also uses them elsewhere holds them)
  context   ``gather_rows_arrays``: the context of each sequence of a step, read
            through its block table from every K and V array
  tier      ``read_block`` per evicted block, ``flush``, ``write_blocks``: evictions to
            pinned host memory and their restore into other blocks

All of them move bytes; only ``write`` with rows of a wider type than the cache
computes anything (the rounding to the cache type).
"""
import math
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path.cwd() / "inference-engine_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from iekv.engine.copier import HipSlotCopier  # noqa: E402
from iekv.engine.pools import KVPool, allocate_pool, allocate_pool_pair  # noqa: E402
from iekv.engine.slots import gather_rows_arrays, write_slots_layers  # noqa: E402

DEVICE = "cuda"
DTYPES = {"float32": torch.float32, "float16": torch.float16, "bfloat16": torch.bfloat16,
          "fp8_e4m3": torch.float8_e4m3fn}
BITS = {1: torch.uint8, 2: torch.int16, 4: torch.int32}

# Pool geometries of the package's benchmark workloads.
SMALL = dict(layers=4, kv_heads=4, head_dim=32, block_size=16, dtype="float32")
QWEN = dict(layers=24, kv_heads=2, head_dim=64, block_size=256, dtype="float16")
LLAMA_8B = dict(layers=32, kv_heads=8, head_dim=128, block_size=16, dtype="bfloat16")
LLAMA_70B = dict(layers=80, kv_heads=8, head_dim=128, block_size=16, dtype="fp8_e4m3")
# A generic model whose tiles are no power of two (five heads of 80).
RAGGED = dict(layers=28, kv_heads=5, head_dim=80, block_size=16, dtype="float16")


def listed():
    return [
        # One short prompt (about 270 tokens) of a small model, handed to the decode pool.
        dict(name="direct_short", op="direct", **SMALL, requests=1, blocks=17, pool=4096),
        # One mean prompt (about 3,090 tokens) of the 8B shape.
        dict(name="direct_8b", op="direct", **LLAMA_8B, requests=1, blocks=193, pool=2048),
        # One 16,384-token prompt of the 70B shape's fp8 share: the largest call.
        dict(name="direct_70b_long", op="direct", **LLAMA_70B, requests=1, blocks=1024,
             pool=1200),
        # A decode worker that keeps its tables on the GPU and has them checked before
        # the move (a 1,000-token prompt of the 8B shape).
        dict(name="checked_8b", op="checked", **LLAMA_8B, requests=1, blocks=63, pool=2048),
        # 64 prompts of 16 to 512 tokens admitted together.
        dict(name="requests_64", op="requests", **SMALL, requests=64, blocks=17, pool=4096),
        # A 400-token prompt through a packed payload (large blocks).
        dict(name="transfer_qwen", op="transfer", **QWEN, requests=1, blocks=2, pool=256),
        # A 1,500-token prompt through a packed payload, tiles of an odd size.
        dict(name="transfer_ragged", op="transfer", **RAGGED, requests=1, blocks=94,
             pool=1500),
        # The KV writes of one decode step over 48 sequences.
        dict(name="write_decode_8b", op="write", **LLAMA_8B, rows="bfloat16", requests=48,
             tokens=1, slots="list", pool=1024),
        # The KV writes of a 3,001-token prefill computed in float32 with a bfloat16 cache.
        dict(name="write_prefill_f32", op="write", **LLAMA_8B, rows="float32", requests=1,
             tokens=3001, slots="device", pool=1024),
        # The contexts of a step over 8 sequences of about 300 tokens each.
        dict(name="context_qwen", op="context", **QWEN, requests=8, tokens=300, pool=256),
        # One 7,777-token context of the 8B shape.
        dict(name="context_8b_long", op="context", **LLAMA_8B, requests=1, tokens=7777,
             pool=1024),
        # 12 blocks evicted to the host tier and restored under other ids.
        dict(name="tier_8b", op="tier", **LLAMA_8B, requests=1, blocks=12, pool=512),
    ]


OPS = ("direct", "checked", "requests", "transfer", "write", "context", "tier")
LARGEST = 2 * 1024 * 160 * 16384          # bytes of direct_70b_long, read and written
STEP_TOKENS = 16384                       # tokens of the longest context or prefill step
# Types a model computes K and V in, by the cache's type.
ROW_TYPES = {"float32": ["float32"], "float16": ["float16", "float32"],
             "bfloat16": ["bfloat16", "float32"], "fp8_e4m3": ["bfloat16", "float32"]}


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Any operation over the listed range of models, table lengths and types."""
    while True:
        c = dict(op=rng.choice(OPS), layers=_log_int(rng, 2, 80),
                 kv_heads=rng.choice([1, 2, 3, 4, 5, 8]),
                 head_dim=rng.choice([32, 64, 80, 96, 128]),
                 block_size=rng.choice([8, 16, 16, 16, 32, 64, 256]),
                 dtype=rng.choice(["float32", "float16", "bfloat16", "fp8_e4m3"]), requests=1)
        if c["op"] == "write":
            c["rows"] = rng.choice(ROW_TYPES[c["dtype"]])
            c["slots"] = rng.choice(["list", "device"])
            c["requests"] = rng.choice([1, 1, 3, 31, 128])
            # One token of each sequence, or a prefill's (lists name a decode step's).
            most = STEP_TOKENS // (8 if c["slots"] == "list" else 1)
            c["tokens"] = 1 if c["requests"] > 3 else _log_int(rng, 1, most // c["requests"])
        elif c["op"] == "context":
            c["requests"] = rng.choice([1, 1, 2, 5, 8])
            c["tokens"] = _log_int(rng, 1, STEP_TOKENS)
        else:
            if c["op"] == "requests":
                c["requests"] = rng.choice([2, 7, 16, 64])
            c["blocks"] = _log_int(rng, 1, 256 if c["op"] == "tier" else 1024)
        blocks = sum(_blocks(c))
        c["pool"] = int(blocks * rng.uniform(1.2, 4)) + 8
        if c["op"] == "tier":
            c["pool"] += blocks                  # evicted and restored blocks are disjoint
        # Bytes over the host link count for what they take there.
        cost = work(c)["bytes"] * (60 if c["op"] == "tier" else 1)
        if cost <= LARGEST and 2 * _pool_bytes(c) <= 16e9 and blocks <= 16384:
            return c


def _row(case):
    return case["kv_heads"] * case["head_dim"]


def _size(case):
    return torch.empty(0, dtype=DTYPES[case["dtype"]]).element_size()


def _pool_bytes(case):
    return 2 * case["layers"] * case["pool"] * case["block_size"] * _row(case) * _size(case)


def _counts(case):
    """Blocks (or tokens) of each request: all alike for one, spread around the mean for more."""
    n, mean = case["requests"], case["blocks"] if "blocks" in case else case["tokens"]
    return [max(1, round(mean * (0.2 + 1.6 * (k + 0.5) / n))) if n > 1 and mean > 1 else mean
            for k in range(n)]


def _blocks(case):
    """Blocks of each request's table."""
    return [-(-c // case["block_size"]) if "tokens" in case else c for c in _counts(case)]


def _generator(seed, device=DEVICE):
    gen = torch.Generator(device=device)
    gen.manual_seed(seed)
    return gen


def _fill(t, gen):
    """N(0,1) values; for fp8 random codes without its two NaNs (the bytes a cache holds)."""
    if t.element_size() == 1:
        raw = t.view(torch.uint8)
        raw.random_(0, 127, generator=gen)
        raw.bitwise_or_((torch.rand(raw.shape, device=raw.device, generator=gen,
                                    dtype=torch.float16) < 0.5).to(torch.uint8) * 128)
    else:
        t.normal_(generator=gen)


def _tables(case, seed, pools):
    """``pools`` lists of block tables, one per request: random blocks, none twice in a pool."""
    gen, out = _generator(seed, "cpu"), []
    for _ in range(pools):
        ids = torch.randperm(case["pool"], generator=gen).tolist()
        at, tables = 0, []
        for c in _blocks(case):
            tables.append(ids[at:at + c])
            at += c
        out.append(tables)
    return out


def _slots(case, seed):
    """The slot of every token of the step: decode steps append one token to each sequence,
    a prefill fills its blocks from the start."""
    bs = case["block_size"]
    gen = _generator(seed + 1, "cpu")
    slots = []
    for table, n in zip(_tables(case, seed, 1)[0], _counts(case)):
        if n == 1:
            slots.append(table[0] * bs + int(torch.randint(bs, (1,), generator=gen)))
        else:
            slots += [table[i // bs] * bs + i % bs for i in range(n)]
    return slots


def _step_rows(case, seed):
    n = sum(_counts(case))
    gen = _generator(seed + 2)
    shape = (case["layers"], n, case["kv_heads"], case["head_dim"])
    return [torch.randn(shape, device=DEVICE, generator=gen).to(DTYPES[case["rows"]])
            for _ in range(2)]


def _slab(caches):
    """The whole memory of a pool's K and V caches as one tensor [2, L, slots, H, D]."""
    k, v = caches
    first = k[0]
    half = (v[0].data_ptr() - first.data_ptr()) // first.element_size()
    layer = first.numel()
    return first.as_strided((2, len(k), *first.shape), (half, layer, *first.stride()))


def prepare(case, seed):
    dims = (case["block_size"], case["layers"], case["kv_heads"], case["head_dim"])
    dtype, bs = DTYPES[case["dtype"]], case["block_size"]
    op = case["op"]
    if op in ("direct", "checked", "requests", "transfer"):
        src, dst = allocate_pool_pair(case["pool"], case["pool"], *dims, dtype=dtype,
                                      device=DEVICE)
        _fill(_slab(src), _generator(seed))
        source = HipSlotCopier(*src, bs)
        dest = HipSlotCopier(*dst, bs, check_device_ids=op == "checked")
        s, d = _tables(case, seed, 2)
        if op == "checked":
            s, d = ([torch.tensor(t, dtype=torch.int32, device=DEVICE) for t in x]
                    for x in (s, d))
        return dict(op=op, source=source, dest=dest, tables=list(zip(s, d)), out=_slab(dst))
    caches = allocate_pool(case["pool"], *dims, dtype=dtype, device=DEVICE)
    if op == "write":
        slots = _slots(case, seed)
        if case["slots"] == "device":
            slots = torch.tensor(slots, dtype=torch.int64, device=DEVICE)
        return dict(op=op, pool=KVPool(*caches, bs), rows=_step_rows(case, seed), slots=slots,
                    out=_slab(caches))
    _fill(_slab(caches), _generator(seed))
    if op == "context":
        return dict(op=op, pool=KVPool(*caches, bs), tables=_tables(case, seed, 1)[0],
                    lengths=_counts(case))
    both = _tables(dict(case, blocks=2 * case["blocks"]), seed, 1)[0][0]
    return dict(op=op, copier=HipSlotCopier(*caches, bs, payload_location="host",
                                            defer_reads=True),
                evicted=both[:case["blocks"]], restored=both[case["blocks"]:],
                out=_slab(caches))


def _values(t):
    """A cache as it is compared: fp8 as its codes."""
    return t.view(torch.uint8) if t.element_size() == 1 else t


def run(state):
    op = state["op"]
    if op in ("direct", "checked"):
        for s, d in state["tables"]:
            state["dest"].copy_blocks(state["source"], s, d)
        return _values(state["out"])
    if op == "requests":
        state["dest"].copy_requests(state["source"], state["tables"])
        return _values(state["out"])
    if op == "transfer":
        payloads = []
        for s, d in state["tables"]:
            packed = state["source"].read_blocks(s)
            state["dest"].write_blocks(d, packed)
            payloads.append(packed.data)
        return [_values(state["out"]), payloads]
    if op == "write":
        write_slots_layers(state["pool"], *state["rows"], state["slots"])
        return _values(state["out"])
    if op == "context":
        return [_values(gather_rows_arrays(state["pool"], t, n))
                for t, n in zip(state["tables"], state["lengths"])]
    payloads = [state["copier"].read_block(b) for b in state["evicted"]]
    state["copier"].flush()
    state["copier"].write_blocks(state["restored"], payloads)
    return _values(state["out"])


def work(case):
    """Bytes read and written; ids and slots are left out (thousands of times smaller)."""
    arrays, row = 2 * case["layers"], _row(case)
    size, n = _size(case), sum(_counts(case))
    if case["op"] == "write":
        wide = torch.empty(0, dtype=DTYPES[case["rows"]]).element_size()
        return {"bytes": arrays * n * row * (wide + size), "flops": 0}
    if case["op"] == "context":
        return {"bytes": 2 * arrays * n * row * size, "flops": 0}
    moved = arrays * n * case["block_size"] * row * size
    # A transfer's payload and a tier's host images are written, then read.
    return {"bytes": moved * (4 if case["op"] in ("transfer", "tier") else 2), "flops": 0}


def tolerance(case):
    """Copies are exact, and a cast to the cache type rounds to nearest even: one right
    result, bit for bit."""
    return "exact"


def exact(case, seed):
    """The same in plain torch: the moved bytes as 64-bit values, and float rows as they were
    before the cache's rounding. fp8 codes are whole numbers that have no such value."""
    if case["dtype"] == "fp8_e4m3" or 4 * _pool_bytes(case) > 40e9:
        return None
    op, bs = case["op"], case["block_size"]
    dtype = DTYPES[case["dtype"]]
    shape = (2, case["layers"], case["pool"] * bs, case["kv_heads"], case["head_dim"])
    src = torch.zeros(shape, dtype=dtype, device=DEVICE)
    if op == "write":
        out = src.double()
        slots = torch.tensor(_slots(case, seed), device=DEVICE)
        for half, rows in zip(out, _step_rows(case, seed)):
            half[:, slots] = rows.double()
        return out
    _fill(src, _generator(seed))
    blocks = src.double().view(2, case["layers"], case["pool"], bs, *shape[3:])
    if op == "context":
        return [blocks[:, :, t].flatten(2, 3)[:, :, :n].flatten(0, 1)
                for t, n in zip(_tables(case, seed, 1)[0], _counts(case))]
    if op == "tier":
        both = _tables(dict(case, blocks=2 * case["blocks"]), seed, 1)[0][0]
        s, d = [both[:case["blocks"]]], [both[case["blocks"]:]]
        out = blocks
    else:
        s, d = _tables(case, seed, 2)
        out = torch.zeros_like(blocks)
    for a, b in zip(s, d):
        out[:, :, b] = blocks[:, :, a]
    out = out.view(shape)
    return [out, [None] * len(s)] if op == "transfer" else out
