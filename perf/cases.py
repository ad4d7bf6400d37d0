"""Performance cases of the KV migration path, through its public entry points.

A case is a dict of plain values; `kind` says which part of a serving program
it stands for:

  append   a step's new K/V rows go into the paged cache, layer by layer:
           decode (one token per request; eager, or replayed from a HIP graph
           as a serving loop does) and prefill (whole prompts), in the fused
           form or in FlashInfer's form with positions computed once per step
  promote  KVMigrator.promote of a batch of requests from one instance's pool
           to another's: through a transfer buffer, fused, or through pinned
           host memory; the destination pages are freed afterwards, as when
           the promoted requests end
  move     KVMigrator.move_pages, the same movement for a program that keeps
           its block tables on the device
  pack     KVhelper.pack_pages and unpack_pages with host block tables: a
           request's pages through a device-resident buffer
  dropin   KVhelper.get_kv_cache and insert_kv_cache: the reference's worker
           calls, through host memory
  swap     SwapSpace.swap_out and swap_in of one preempted request

All of them move data and compute nothing, so outputs are exact.
"""
import math
from types import SimpleNamespace

import numpy as np
import torch

from paceserve_amd.core.block_manager import NativeBlockAllocator
from paceserve_amd.kv_transfer import append as kv_append
from paceserve_amd.kv_transfer.kv_utils import KVhelper
from paceserve_amd.kv_transfer.migrate import KVMigrator
from paceserve_amd.kv_transfer.swap import SwapSpace

DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16, "float32": torch.float32,
          "float8_e4m3fn": torch.float8_e4m3fn}
ELEM = {"float16": 2, "bfloat16": 2, "float32": 4, "float8_e4m3fn": 1}
LLAMA3 = dict(heads=8, head_dim=128, page=16, dtype="bfloat16")
LLAMA3_TP8 = dict(LLAMA3, heads=1)     # one GPU's KV head at tensor parallelism 8
LLAMA2_7B = dict(LLAMA3, heads=32, dtype="float16")
MiB = 1 << 20


def listed():
    return [
        # A decode step of 256 running requests, replayed from a graph: the
        # launches are tiny and follow one another, one per layer.
        dict(LLAMA3, name="decode_256req_graph", kind="append", layers=32, requests=256, tokens=1, ragged=False,
             context=128, fused=True, graph=True, strided=False),
        # A prefill batch; K and V are slices of the fused QKV projection.
        dict(LLAMA3, name="prefill_16x1024", kind="append", layers=1, requests=16, tokens=1024, ragged=False,
             context=0, fused=True, graph=False, strided=True),
        # A long prompt on one GPU of a tensor-parallel group: 256-byte rows.
        dict(LLAMA3_TP8, name="prefill_32768_tp8", kind="append", layers=1, requests=1, tokens=32768, ragged=False,
             context=0, fused=True, graph=False, strided=False),
        # Multi-head attention without grouped KV heads: 8 KiB rows; chunked
        # prefill continues prompts at unaligned positions.
        dict(LLAMA2_7B, name="prefill_2x4095_7b", kind="append", layers=4, requests=2, tokens=4095, ragged=False,
             context=777, fused=False, graph=False, strided=False),
        # The shortest request, where launch latency is all.
        dict(LLAMA3, name="promote_16tok", kind="promote", layers=32, requests=1, tokens=16, mode="buffer",
             extra=True),
        # One 512-token request by host block tables.
        dict(LLAMA3, name="pack_unpack_512tok", kind="pack", layers=32, requests=1, tokens=512, dtype="float16"),
        # One long request.
        dict(LLAMA3, name="promote_4096tok", kind="promote", layers=32, requests=1, tokens=4096, mode="buffer",
             extra=False),
        # A batch on one GPU of a tensor-parallel group: 8 KiB pages, 80 layers.
        dict(LLAMA3_TP8, name="promote_64req_tp8", kind="promote", layers=80, requests=64, tokens=2048,
             mode="buffer", extra=False),
        # Pages of a single token: 512 bytes, half a wavefront's vectors.  Tables
        # of thousands of entries stay on the device.
        dict(LLAMA3_TP8, name="move_4req_page1_tp8", kind="move", layers=32, requests=4, tokens=4096, page=1,
             mode="fused"),
        # The host legs.
        dict(LLAMA3, name="promote_4096tok_pinned", kind="promote", layers=32, requests=1, tokens=4096,
             mode="pinned", extra=False),
        dict(LLAMA3, name="dropin_100tok", kind="dropin", layers=32, requests=1, tokens=100),
        dict(LLAMA3, name="swap_1024tok", kind="swap", layers=32, requests=1, tokens=1000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a KV shape, then a batch whose payload fits the kind's
    range (at most what the largest listed case of its kind moves)."""
    while True:
        kind = rng.choice(["append", "append", "append", "promote", "promote", "move", "move", "pack", "dropin",
                           "swap"])
        c = dict(kind=kind, heads=rng.choice([1, 2, 3, 4, 5, 8, 12, 16, 32]),
                 head_dim=rng.choice([64, 80, 96, 112, 128, 192, 256]), page=rng.choice([1, 4, 8, 16, 16, 32, 64]),
                 dtype=rng.choice(list(DTYPES)))
        if kind == "append":
            decode = rng.random() < 0.4
            c.update(layers=_log_int(rng, 1, 48) if decode else _log_int(rng, 1, 4),
                     requests=_log_int(rng, 1, 512) if decode else _log_int(rng, 1, 32),
                     tokens=1 if decode else _log_int(rng, 16, 32768), ragged=not decode and rng.random() < 0.7,
                     context=rng.randrange(0, 300), fused=rng.random() < 0.6,
                     graph=decode and rng.random() < 0.6, strided=rng.random() < 0.4)
            lo, hi = 0, 256 * MiB
        else:
            c.update(layers=_log_int(rng, 4, 80), requests=_log_int(rng, 1, 64) if kind in ("promote", "move") else 1,
                     tokens=_log_int(rng, 10, 8192))
            if kind in ("promote", "move"):
                c.update(mode=rng.choice(["buffer", "buffer", "fused", "fused", "pinned"]))
            if kind == "promote":
                c.update(extra=rng.random() < 0.3)
            lo, hi = 64 << 10, 2048 * MiB
            if kind in ("dropin", "swap") or c.get("mode") == "pinned":
                hi = 256 * MiB
        if lo <= _payload(c) <= hi and _cache_bytes(c) <= 4096 * MiB:
            return c


# ------------------------------------------------------------------- sizes

def _ceil(a, b):
    return -(-a // b)


def _row_bytes(c):
    return c["heads"] * c["head_dim"] * ELEM[c["dtype"]]


def _page_bytes(c):
    return 2 * c["page"] * _row_bytes(c)


def _lengths(c):
    """Tokens of each request: the case's for one request, spread between a
    32nd of it and all of it for a batch; an append's are equal unless ragged."""
    n, t = c["requests"], c["tokens"]
    if c["kind"] == "append" and not c["ragged"]:
        return [t] * n
    if n == 1:
        return [t]
    return [max(1, t - int(i * 0.6180339887 % 1.0 * (t - t // 32))) for i in range(n)]


def _priors(c):
    """Tokens each request of an append already holds."""
    return [int((0.5 + i * 0.6180339887) % 1.0 * c["context"]) for i in range(c["requests"])]


def _request_pages(c):
    if c["kind"] == "append":
        return [_ceil(a + b, c["page"]) for a, b in zip(_lengths(c), _priors(c))]
    return [_ceil(n, c["page"]) for n in _lengths(c)]


def _pool_pages(c):
    """A pool somewhat larger than what the batch holds (and the extra page
    of each request that opens one); a swapped request comes back to other
    pages of the same pool."""
    n = sum(_request_pages(c)) + c["requests"]
    return 2 * n if c["kind"] == "swap" else n + n // 4 + 7


def _payload(c):
    if c["kind"] == "append":
        return 2 * c["layers"] * sum(_lengths(c)) * _row_bytes(c)
    return c["layers"] * sum(_request_pages(c)) * _page_bytes(c)


def _cache_bytes(c):
    return c["layers"] * _pool_pages(c) * _page_bytes(c)


def work(case):
    """Each payload byte is read once and written once per copy the caller
    asks for: an append or a fused movement is one copy; pack, dropin, swap
    and the movements through a buffer are two, since the buffer between
    them, which holds the request's payload, is a result of its own."""
    copies = 1 if case["kind"] == "append" or case.get("mode") == "fused" else 2
    return {"bytes": 2 * copies * _payload(case), "flops": 0}


def tolerance(case):
    return "exact"


# ------------------------------------------------------------------ inputs

def _random(shape, case, gen):
    dtype = DTYPES[case["dtype"]]
    t = torch.empty(shape, dtype=torch.bfloat16 if ELEM[case["dtype"]] == 1 else dtype, device="cuda")
    t.normal_(generator=gen)
    return t if t.dtype == dtype else t.to(dtype)


def _cache(case, gen):
    """[layers, pages, 2, page, heads, head_dim]; a layer's cache is its slice."""
    shape = (case["layers"], _pool_pages(case), 2, case["page"], case["heads"], case["head_dim"])
    return _random(shape, case, gen)


def _tables(case, rng, counts):
    """Block tables of a fragmented pool, and the rest of its free list."""
    perm = rng.permutation(_pool_pages(case)).tolist()
    tables = []
    for n in counts:
        tables.append(perm[:n])
        del perm[:n]
    return tables, perm


def _append_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    s = SimpleNamespace(cache=_cache(case, gen))
    H, D = case["heads"], case["head_dim"]
    lengths, priors, pages = _lengths(case), _priors(case), _request_pages(case)
    nnz = sum(lengths)
    s.keys, s.values = [], []
    for _ in range(case["layers"]):
        if case["strided"]:    # query heads, then K and V, of one projection
            qkv = _random((nnz, 4 * H, D), case, gen)
            s.keys.append(qkv[:, 2 * H:3 * H])
            s.values.append(qkv[:, 3 * H:])
        else:
            s.keys.append(_random((nnz, H, D), case, gen))
            s.values.append(_random((nnz, H, D), case, gen))
    tables, _ = _tables(case, rng, pages)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    s.append_indptr = i32(np.concatenate([[0], np.cumsum(lengths)]))
    s.kv_indptr = i32(np.concatenate([[0], np.cumsum(pages)]))
    s.kv_indices = i32(sum(tables, []))
    s.last = i32([(a + b - 1) % case["page"] + 1 for a, b in zip(lengths, priors)])
    s.nnz, s.tables, s.lengths, s.priors = nnz, tables, lengths, priors
    return s


def _pool_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.default_rng(seed)
    pages = _request_pages(case)
    s = SimpleNamespace(src=_cache(case, gen))
    s.dst = s.src if case["kind"] == "swap" else _cache(case, gen)
    s.src_tables, rest = _tables(case, rng, pages)
    if case["kind"] == "swap":
        s.dst_tables = [rest[:pages[0]]]
        return s
    s.dst_free = rng.permutation(_pool_pages(case)).tolist()
    s.dst_counts = [n + 1 for n in pages] if case.get("extra") else None
    free, s.dst_tables = list(s.dst_free), []
    for n in s.dst_counts or pages:     # the last free page goes first
        s.dst_tables.append([free.pop() for _ in range(n)])
    return s


def _helper(case, cache):
    H, D = case["heads"], case["head_dim"]
    model = SimpleNamespace(get_num_q_heads=lambda p: 4 * H, get_num_kv_heads=lambda p: H, get_head_size=lambda: D,
                            dtype=DTYPES[case["dtype"]], get_num_layers=lambda p: case["layers"])
    h = KVhelper(0, model, SimpleNamespace(block_size=case["page"]), None)
    wrapper = SimpleNamespace(gpu_cache=list(cache))
    h.add_model_runner(SimpleNamespace(attention_backend_wrapper=wrapper))
    return h


def prepare(case, seed):
    if case["kind"] == "append":
        s = _append_inputs(case, seed)
        s.case = case
        if case["graph"]:
            _append_step(s)
            torch.cuda.synchronize()
            s.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s.graph):
                _append_step(s)
        return s
    s = _pool_inputs(case, seed)
    s.case = case
    if case["kind"] in ("promote", "move"):
        s.allocator = NativeBlockAllocator(case["page"], _pool_pages(case), s.dst_free)
        s.migrator = KVMigrator(list(s.src), list(s.dst), s.allocator)
        s.host_buf = None
        if case["mode"] == "pinned":
            s.host_buf = torch.empty(_payload(case), dtype=torch.uint8, pin_memory=True)
        if case["kind"] == "move":
            s.src_ids, s.dst_ids = (torch.tensor(sum(t, []), dtype=torch.int32, device="cuda")
                                    for t in (s.src_tables, s.dst_tables))
    elif case["kind"] == "swap":
        s.space = SwapSpace(list(s.src), len(s.src_tables[0]) + 8)
    else:
        s.from_helper, s.to_helper = _helper(case, s.src), _helper(case, s.dst)
        s.seq = SimpleNamespace(seq_id="0")
        s.seq_manager = SimpleNamespace(_get_block_table=lambda seq: s.src_tables[0])
    return s


# --------------------------------------------------------------------- run

def _append_step(s):
    if s.case["fused"]:
        for l, cache in enumerate(s.cache):
            kv_append.append_paged_kv_cache_indptr(s.keys[l], s.values[l], s.append_indptr, cache, s.kv_indices,
                                                   s.kv_indptr, s.last)
        return
    seq_lens = kv_append.get_seq_lens(s.kv_indptr, s.last, s.case["page"])
    batch, positions = kv_append.get_batch_indices_positions(s.append_indptr, seq_lens, s.nnz)
    for l, cache in enumerate(s.cache):
        kv_append.append_paged_kv_cache(s.keys[l], s.values[l], batch, positions, cache, s.kv_indices, s.kv_indptr,
                                        s.last)


def run(state):
    s, c = state, state.case
    if c["kind"] == "append":
        if c["graph"]:
            s.graph.replay()
        else:
            _append_step(s)
        return {"cache": s.cache}
    if c["kind"] == "promote":
        plan = s.migrator.promote(s.src_tables, s.dst_counts, c["mode"], host_buf=s.host_buf)
        s.allocator.free_many(p for t in reversed(plan.dst_tables) for p in reversed(t))
        return {"dst": s.dst, "pages": np.array(plan.dst_ids, dtype=np.int64)}
    if c["kind"] == "move":
        s.migrator.move_pages(s.src_ids, s.dst_ids, c["mode"], host_buf=s.host_buf)
        return {"dst": s.dst}
    if c["kind"] == "pack":
        buf = s.from_helper.pack_pages(s.src_tables[0])
        s.to_helper.unpack_pages(buf, s.dst_tables[0])
        return {"buffer": buf, "dst": s.dst}
    if c["kind"] == "dropin":
        content, _ = s.from_helper.get_kv_cache(s.seq, s.seq_manager)
        ok = s.to_helper.insert_kv_cache(content, s.dst_tables[0], "cuda")
        return {"content": content, "dst": s.dst, "ok": ok}
    s.space.swap_out("0", s.src_tables[0])
    s.space.swap_in("0", s.dst_tables[0])
    return {"pool": s.dst}


# ------------------------------------------------------------------- exact

def exact(case, seed):
    """The same bytes by torch's own indexing."""
    if case["kind"] == "append":
        s = _append_inputs(case, seed)
        page, slot = [], []
        for table, n, prior in zip(s.tables, s.lengths, s.priors):
            at = np.arange(prior, prior + n)
            page.append(np.asarray(table)[at // case["page"]])
            slot.append(at % case["page"])
        page = torch.from_numpy(np.concatenate(page)).to("cuda")
        slot = torch.from_numpy(np.concatenate(slot)).to("cuda")
        words = lambda t: t.view(torch.uint8) if t.element_size() == 1 else t  # noqa: E731
        for l, cache in enumerate(s.cache):
            words(cache)[page, 0, slot] = words(s.keys[l])
            words(cache)[page, 1, slot] = words(s.values[l])
        return {"cache": s.cache}
    s = _pool_inputs(case, seed)
    src_ids = sum(s.src_tables, [])
    dst_ids = sum((t[:n] for t, n in zip(s.dst_tables, map(len, s.src_tables))), [])
    si, di = torch.tensor(src_ids, device="cuda"), torch.tensor(dst_ids, device="cuda")
    words = (lambda t: t.view(torch.uint8)) if ELEM[case["dtype"]] == 1 else (lambda t: t)
    picked = words(s.src)[:, si]
    words(s.dst)[:, di] = picked
    content = picked.view(DTYPES[case["dtype"]])
    if case["kind"] == "promote":
        return {"dst": s.dst, "pages": np.array(dst_ids, dtype=np.int64)}
    if case["kind"] == "move":
        return {"dst": s.dst}
    if case["kind"] == "pack":
        return {"buffer": content, "dst": s.dst}
    if case["kind"] == "dropin":
        return {"content": content, "dst": s.dst, "ok": True}
    return {"pool": s.dst}
