"""The calls this framework's users make, sized over the range they make them at.

A serving rank uses the library in three ways, and the cases follow them:

- **the snapshot** (``gather``): on every decode step the step's few slots, and on a notice a
  window of thousands of slots or whole blocks, are gathered out of the paged cache into staging
  rows ``[layers, heads, capacity, 2, head_dim]``;
- **the restore** (``scatter``, ``order``, ``tables``): a lost rank's rows go back into a fresh
  paged cache, from staging rows on the device or from the store's host tables;
- **the reduction** (``reduce``, ``slot``): the sum over the members' buffers, at decode sizes
  inside a captured graph (one call for each all-reduce of a step) and at prefill sizes eagerly.

Rows and slot ids are moved, not computed, and the sum's order is part of its definition, so every
output is compared bit for bit.
"""

from __future__ import annotations

import math

import numpy as np
import torch

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "fp8": torch.float8_e4m3fn}
LAYOUTS = ("kv_first", "blocks_first", "combined")
MAX_ROWS = 8
MAX_SLOT_N = 65536  # the slot collective's largest tensor (SlotKernel's MAXN)


def listed():
    return [
        # one decode step of a Llama-3-8B rank: 64 sequences, one new slot each, every layer
        dict(name="snapshot_decode", kind="gather", by="slots", layout="kv_first", dtype="bf16",
             layers=32, heads=8, held=8, head_dim=128, block_size=16, num_blocks=2048, count=64,
             padding=0.0),
        # a window of 16,384 slots of the same rank: the benchmark's headline
        dict(name="snapshot_window", kind="gather", by="slots", layout="kv_first", dtype="bf16",
             layers=32, heads=8, held=8, head_dim=128, block_size=16, num_blocks=8192, count=16384,
             padding=0.0, whole_blocks=True),
        # a notice round by block table, Llama-3-70B on 8 ranks: one fp8 KV head, with slot tags
        dict(name="notice_blocks_fp8", kind="gather", by="blocks", layout="kv_first", dtype="fp8",
             layers=80, heads=1, held=1, head_dim=128, block_size=16, num_blocks=4096, count=2048,
             padding=0.0),
        # half-rows that are no whole number of 16-byte words, a ragged slot list with padding,
        # and a rank that holds half of the cache's head slots
        dict(name="snapshot_odd", kind="gather", by="slots", layout="combined", dtype="fp8",
             layers=36, heads=12, held=6, head_dim=120, block_size=16, num_blocks=1024, count=5001,
             padding=0.02),
        # a restore's rows in staged order, below the size at which the loader sorts first
        dict(name="scatter_staged", kind="scatter", layout="kv_first", dtype="bf16", layers=4,
             heads=8, held=8, head_dim=128, block_size=16, num_blocks=4096, count=65536,
             padding=0.0),
        # a whole cache of 262,144 slots through a permuted block table: the loader sorts first
        dict(name="scatter_whole", kind="scatter", layout="kv_first", dtype="bf16", layers=8,
             heads=8, held=8, head_dim=128, block_size=16, num_blocks=16384, count=262144,
             padding=0.0),
        # the write order of a whole cache's restore, made on the device
        dict(name="order_whole", kind="order", block_size=16, num_blocks=16384, count=262144,
             padding=0.0),
        # a spare's catch-up from the store's host tables: 64 sequences, the last 16 steps (in
        # tables of 8,192 slots: only the written rows are read)
        dict(name="restore_tables", kind="tables", layers=32, heads=8, head_dim=128,
             block_size=16, num_blocks=512, seqs=64, steps=16),
        # the all-reduces of one captured decode step: 32 layers, two each, 16 Ki elements
        dict(name="reduce_decode", kind="reduce", k=8, n=16384, calls=64, captured=True),
        # a 256-token chunk at hidden size 8192, eager
        dict(name="reduce_chunk", kind="reduce", k=8, n=256 * 8192, calls=1, captured=False),
        # a prefill batch of 8192 tokens at hidden size 4096, four members, eager
        dict(name="reduce_prefill", kind="reduce", k=4, n=8192 * 4096, calls=1, captured=False),
        # the slot collective in one captured decode step: 64 calls of 16 Ki elements
        dict(name="slot_decode", kind="slot", k=4, n=16384, calls=64, push=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _rows_bytes(case):
    elem = 1 if case["dtype"] == "fp8" else 2
    n = case["count"] * (case["block_size"] if case.get("by") == "blocks" else 1)
    return case["layers"] * case["held"] * n * 2 * case["head_dim"] * elem


def draw(rng):
    kind = rng.choice(["gather"] * 5 + ["scatter"] * 3 + ["order", "tables"] + ["reduce"] * 3
                      + ["slot"])
    if kind == "order":
        count = _log_int(rng, 1024, 1 << 20)
        blocks = -(-count // 16) * rng.choice([1, 1, 2, 3]) + rng.randrange(8)
        return dict(kind=kind, block_size=16, num_blocks=blocks, count=count,
                    padding=rng.choice([0.0, 0.01]))
    if kind == "tables":
        return dict(kind=kind, layers=rng.choice([8, 16, 28, 32]), heads=rng.choice([2, 4, 8]),
                    head_dim=rng.choice([64, 128]), block_size=16, num_blocks=512,
                    seqs=rng.randrange(8, 65), steps=rng.randrange(4, 33))
    if kind == "reduce":
        k = rng.randrange(1, MAX_ROWS + 1)
        if rng.random() < 0.4:
            return dict(kind=kind, k=k, n=_log_int(rng, 1024, 131072), calls=rng.randrange(32, 97),
                        captured=True)
        return dict(kind=kind, k=k, n=_log_int(rng, 131072, 1 << 25), calls=1, captured=False)
    if kind == "slot":
        return dict(kind=kind, k=rng.randrange(1, MAX_ROWS + 1),
                    n=2 * _log_int(rng, 512, MAX_SLOT_N // 2), calls=rng.randrange(32, 97),
                    push=rng.random() < 0.5)
    heads = rng.choice([1, 2, 4, 8, 12])
    case = dict(kind=kind, layout=rng.choice(LAYOUTS), dtype=rng.choice(["bf16", "bf16", "f16", "fp8"]),
                layers=rng.choice([1, 4, 16, 24, 28, 32, 40, 80]), heads=heads,
                held=rng.choice([heads, heads, max(1, heads // 2)]),
                head_dim=rng.choice([64, 80, 96, 112, 120, 128, 128, 192, 256]),
                block_size=16, padding=rng.choice([0.0, 0.0, 0.02]))
    if kind == "gather":
        case["by"] = rng.choice(["slots", "slots", "blocks"])
        case["count"] = _log_int(rng, 1, 16384) if case["by"] == "slots" else _log_int(rng, 1, 1024)
        if case["by"] == "blocks":
            case["padding"] = 0.0
    else:
        case["count"] = _log_int(rng, 64, 131072)
    # half-rows that are no whole number of 16-byte words cost more a byte
    ragged = case["head_dim"] * (1 if case["dtype"] == "fp8" else 2) % 16 != 0
    while _rows_bytes(case) > (256 << 20 if ragged else 2 << 30) and case["count"] > 1:
        case["count"] = case["count"] // 2 + case["count"] % 2
    blocks = case["count"] if case.get("by") == "blocks" else -(-case["count"] // 16)
    case["num_blocks"] = blocks + max(8, blocks // rng.choice([1, 2, 4]))
    return case


def _shape(layout, blocks, block_size, heads, d):
    return {"kv_first": (2, blocks, block_size, heads, d),
            "blocks_first": (blocks, 2, block_size, heads, d),
            "combined": (blocks, heads, block_size, 2 * d)}[layout]


def _values(shape, dtype, g):
    """N(0, 1) rows; for fp8 what a scale of 1/20 leaves of them, saturated at e4m3's range."""
    if dtype is torch.float8_e4m3fn:
        x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float16)
        return x.mul_(20).clamp_(-448, 448).to(dtype)
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(generator=g)


def _slots(case, rng, count=None):
    """``count`` distinct slots: whole blocks of a permuted block table, or (a decode step) one
    slot in each of that many blocks while there are enough; some of them padding."""
    bs, nb = case["block_size"], case["num_blocks"]
    count = case["count"] if count is None else count
    if case["kind"] == "gather" and not case.get("whole_blocks") and count * 2 <= nb:
        s = rng.permutation(nb)[:count] * bs + rng.integers(0, bs, count)
    else:
        need = -(-count // bs)
        s = (rng.permutation(nb)[:need, None] * bs + np.arange(bs)[None, :]).reshape(-1)[:count]
    s = s.astype(np.int64)
    if case["padding"]:
        s[rng.random(count) < case["padding"]] = -1
    return s


def _paged(case, fill, g):
    from everserve_amd.state.paged import PagedKV

    dtype = DTYPES[case.get("dtype", "bf16")]
    shape = _shape(case.get("layout", "kv_first"), case["num_blocks"], case["block_size"],
                   case["heads"], case["head_dim"])
    caches = torch.zeros((case["layers"], *shape), dtype=dtype, device="cuda")
    if fill:
        for t in caches:
            t.copy_(_values(shape, dtype, g))
    ptrs = torch.tensor([t.data_ptr() for t in caches], dtype=torch.long, device="cuda")
    strides = list(PagedKV.of(caches[0]).layout_strides(caches[0]))
    return caches, ptrs, strides, dtype


def _written(case, rng):
    """The slots a decode run wrote in its last ``steps`` steps, as sorted (start, count) ranges."""
    bs, nb, seqs = case["block_size"], case["num_blocks"], case["seqs"]
    table = rng.permutation(nb)[:seqs * (nb // seqs)].reshape(seqs, nb // seqs)
    first = rng.integers(0, (nb // seqs) * bs - case["steps"], seqs)
    pos = first[:, None] + np.arange(case["steps"])[None, :]
    slots = np.sort((table[np.arange(seqs)[:, None], pos // bs] * bs + pos % bs).reshape(-1))
    cut = np.flatnonzero(np.diff(slots) != 1) + 1
    starts, ends = slots[np.r_[0, cut]], slots[np.r_[cut - 1, slots.size - 1]]
    return slots, [(int(a), int(b - a + 1)) for a, b in zip(starts, ends)]


def _members(case, seed):
    """The members' payloads of every call, N(0, 1): a list of calls of lists of k tensors."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [[torch.randn(case["n"], generator=g, device="cuda").to(torch.bfloat16)
             for _ in range(case["k"])] for _ in range(case["calls"])]


def prepare(case, seed):
    from everserve_amd import kernels

    ext = kernels.load()
    kind = case["kind"]
    rng = np.random.default_rng(seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    st = dict(case=case, ext=ext)
    if kind in ("gather", "scatter"):
        caches, ptrs, strides, dtype = _paged(case, kind == "gather", g)
        elem = caches[0].element_size()
        heads = torch.from_numpy(rng.permutation(case["heads"])[:case["held"]].astype(np.int64)).cuda()
        rows = case["count"]
        if case.get("by") == "blocks":
            ids = rng.permutation(case["num_blocks"])[:rows].astype(np.int32)
            rows *= case["block_size"]
            st["tags"] = torch.empty(rows, dtype=torch.long, device="cuda")
        else:
            ids = _slots(case, rng)
        # the staging capacity of a step: a power of two, 8 at least
        cap = max(8, 1 << (rows - 1).bit_length())
        shape = (case["layers"], case["held"], cap, 2, case["head_dim"])
        if kind == "gather":
            staged = torch.zeros(shape, dtype=dtype, device="cuda")
        else:
            staged = _values(shape, dtype, g)
        st.update(caches=caches, staged=staged, ids=torch.from_numpy(ids).cuda(),
                  args=(ptrs, heads, staged.data_ptr(), cap, case["head_dim"], case["block_size"],
                        strides, elem))
    elif kind == "order":
        slots = torch.from_numpy(_slots(case, rng)).cuda()
        st.update(slots=slots, out=(torch.empty_like(slots), torch.empty_like(slots)))
    elif kind == "tables":
        from everserve_amd.state.restore import Restorer, Table

        caches = list(_paged(case, False, g)[0])
        slots, written = _written(case, rng)
        row = 2 * case["head_dim"]
        per_layer = [rng.integers(0, 1 << 16, (slots.size, row), dtype=np.uint16) & 0xBFFF
                     for _ in range(4)]
        tables = []
        for layer in range(case["layers"]):
            for h in range(case["heads"]):
                t = layer * 1000 + h
                x = np.zeros((case["num_blocks"] * case["block_size"], row), dtype=np.uint16)
                x[slots] = per_layer[t % 4] ^ np.uint16(t & 0x3FFF)
                tables.append(Table(t, x.view(np.uint8).reshape(-1), written))
        st.update(caches=caches, tables=tables, restorer=Restorer(ext, caches, freeze_heap=False),
                  head_map={h: (h + 3) % case["heads"] for h in range(case["heads"])})
    else:
        st["members"] = _members(case, seed) if kind == "reduce" else _inputs(case, seed)
        # each call's output starts at a multiple of 128 bytes
        pitch = -(-case["n"] // 64) * 64
        st["out"] = torch.zeros((case["calls"], pitch), dtype=torch.bfloat16,
                                device="cuda")[:, :case["n"]]
        st["outs"] = list(st["out"].unbind(0))
        if kind == "reduce":
            pad = [0] * (MAX_ROWS - case["k"])
            order = [case["k"], *rng.permutation(case["k"]).tolist(), *pad]
            st.update(bufs=[torch.tensor([t.data_ptr() for t in call] + pad, dtype=torch.long,
                                         device="cuda") for call in st["members"]],
                      flags=torch.ones(MAX_ROWS, dtype=torch.long, device="cuda"),
                      order=torch.tensor(order, dtype=torch.int32, device="cuda"),
                      status=torch.zeros(kernels.REDUCE_STATE_WORDS, dtype=torch.long,
                                         device="cuda"))
        else:
            # one GPU has no peer: the listed members are this member's own row, k times over
            words = torch.zeros((2 * MAX_ROWS if case["push"] else 2) * MAX_SLOT_N // 2,
                                dtype=torch.long, device="cuda")
            st.update(words=words,
                      bufs=torch.tensor([words.data_ptr()] * MAX_ROWS, dtype=torch.long,
                                        device="cuda"),
                      ctrl=torch.zeros(MAX_ROWS * ext.CTRL_WORDS, dtype=torch.long, device="cuda"),
                      order=torch.tensor([case["k"]] + [0] * MAX_ROWS, dtype=torch.int32,
                                         device="cuda"),
                      seqs=torch.zeros(ext.slot_blocks(MAX_SLOT_N, 1) + 1, dtype=torch.long,
                                       device="cuda"))
        if case.get("captured", True):
            _all_reduces(st)  # eagerly first, as an engine does before it captures
            torch.cuda.synchronize()
            st["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(st["graph"]):
                _all_reduces(st)
    return st


def _all_reduces(state):
    case, ext = state["case"], state["ext"]
    if case["kind"] == "reduce":
        for bufs, out in zip(state["bufs"], state["outs"]):
            ext.local_reduce(bufs, state["flags"], state["order"], out, 1, 10**9, 0,
                             state["status"])
    else:
        for x, out in zip(state["members"], state["outs"]):
            ext.slot_all_reduce(x, out, state["bufs"], state["ctrl"].data_ptr(), state["order"],
                                state["seqs"], 0, MAX_SLOT_N, 1, case["push"])


def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(case["n"], generator=g, device="cuda").to(torch.bfloat16)
            for _ in range(case["calls"])]


def _bits(t):
    return t.view(torch.uint8) if t.dtype is torch.float8_e4m3fn else t


def run(state):
    case, ext = state["case"], state["ext"]
    kind = case["kind"]
    if kind == "gather":
        ptrs, *rest = state["args"]
        if case["by"] == "blocks":
            ext.gather_blocks(ptrs, state["ids"], *rest, state["tags"])
            return _bits(state["staged"]), state["tags"]
        ext.gather_rows(ptrs, state["ids"], *rest)
        return _bits(state["staged"])
    if kind == "scatter":
        ptrs, *rest = state["args"]
        ext.scatter_rows(ptrs, state["ids"], *rest)
        return _bits(state["caches"])
    if kind == "order":
        return ext.order_pairs(state["slots"], case["num_blocks"] * case["block_size"],
                               out=state["out"])
    if kind == "tables":
        state["restorer"].restore(state["tables"], state["head_map"])
        return state["caches"]
    if "graph" in state:
        state["graph"].replay()
    else:
        _all_reduces(state)
    return state["out"]


def work(case):
    kind = case["kind"]
    if kind in ("gather", "scatter"):
        elem = 1 if case["dtype"] == "fp8" else 2
        n = case["count"] * (case["block_size"] if case.get("by") == "blocks" else 1)
        rows = case["layers"] * case["held"] * n
        return {"bytes": 2 * rows * 2 * case["head_dim"] * elem + n * 8, "flops": 0}
    if kind == "order":
        return {"bytes": 24 * case["count"], "flops": 0}
    if kind == "tables":
        rows = case["layers"] * case["heads"] * case["seqs"] * case["steps"]
        return {"bytes": 2 * rows * 4 * case["head_dim"], "flops": 0}
    members = case["k"] if kind == "reduce" else 1
    return {"bytes": case["calls"] * (members + 1) * case["n"] * 2,
            "flops": case["calls"] * case["k"] * case["n"]}


def tolerance(case):
    # rows and ids are moved, and the sum's order and rounding are its definition
    return "exact"


def exact(case, seed):
    if case["kind"] == "reduce":
        out = torch.zeros((case["calls"], case["n"]), dtype=torch.float64, device="cuda")
        for acc, call in zip(out, _members(case, seed)):
            for t in call:
                acc += t.double()
        return out
    if case["kind"] == "slot":
        return torch.stack([x.double() * case["k"] for x in _inputs(case, seed)])
    return None  # moved bytes and slot ids: no computed number
