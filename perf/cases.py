"""Performance cases of the paged-KV data path, through its public entry points.

A case is one call (or one layer's calls) of a serving program: writing new
K/V rows into pages, gathering sequences, decode attention, prompt attention,
copy-on-write of shared pages, moving chunks between GPU and CPU. The `kind`
picks the calls; the other fields are the cache's shape and the batch. Sequence
lengths come from the case alone (field `lens` seeds them), so the work of a
case is the same for every set of inputs; values and page placement come from
the seed. Pages are always placed at random in the pool, as a pool that has
served requests for a while has them.

Kinds
  write          kvflux_write_paged_kv: `tokens` new rows at their slots
  gather         kvflux_gather_paged_kv_live: `rows` sequences to packed K/V
  decode         kvflux_paged_attention over a batch; with `append`, the
                 step's K/V rows are first written through
                 kvflux_write_paged_kv_tail (one layer of a decode step)
  decode_api     v2.paged_attention_batch over a DeviceBatchTable (the
                 synchronous C++ API, validation and wait included)
  prefill_batch  kvflux_paged_prefill_batch: whole prompts, one launch
  prefill_chunk  kvflux_paged_prefill_split: `new` tokens after a prefix
  prefill_api    v2.paged_attention with its defaults (1e-5 contract) on a
                 whole prompt
  cow            kvflux_copy_pages: `pairs` shared pages copied
  offload        v3.GpuCpuTransfer: a batch of chunks to the CPU and back
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

TORCH = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
CODE = {"f16": 0, "bf16": 1, "f32": 2}
API_DTYPE = {"f16": "Float16", "bf16": "BFloat16", "f32": "Float32"}
BYTES = {"f16": 2, "bf16": 2, "f32": 4}


def _shape(dtype, q_heads, kv_heads, head_size, block_size):
    return {"dtype": dtype, "q_heads": q_heads, "kv_heads": kv_heads, "head_size": head_size,
            "block_size": block_size}


def listed():
    gqa = _shape("bf16", 32, 8, 128, 16)
    return [
        # A few interactive requests: the smallest call of a serving loop,
        # where launches and the wait set the time.
        {"name": "decode_api_4", "kind": "decode_api", **gqa, "rows": 4, "lo": 100, "hi": 1500, "lens": 1},
        # A long prompt's K/V rows going into their pages.
        {"name": "write_4096", "kind": "write", **gqa, "tokens": 4096},
        # Sequences read back into packed form (export, resharding, checks).
        {"name": "gather_64", "kind": "gather", **_shape("f16", 32, 8, 128, 16), "rows": 64, "lo": 512, "hi": 8192,
         "lens": 2},
        # One layer of an ordinary decode step: new rows written, then
        # attention; an odd GQA group and ragged lengths.
        {"name": "decode_layer_16", "kind": "decode", **_shape("f16", 28, 4, 128, 16), "rows": 16, "lo": 512,
         "hi": 8192, "lens": 3, "prefix": 0, "append": True},
        # Two users with long documents: little batch, much context, larger pages.
        {"name": "decode_long_2", "kind": "decode", **_shape("bf16", 32, 8, 128, 32), "rows": 2, "lo": 40000,
         "hi": 70000, "lens": 4, "prefix": 0, "append": False},
        # A full batch behind a shared system prompt: the largest decode.
        {"name": "decode_batch_128", "kind": "decode", **gqa, "rows": 128, "lo": 1024, "hi": 32768, "lens": 5,
         "prefix": 2048, "append": False},
        # A batch of whole prompts.
        {"name": "prefill_8x4096", "kind": "prefill_batch", **gqa, "rows": 8, "lo": 4096, "hi": 4096, "lens": 6},
        # Chunked prefill: the next 512 tokens of a long prompt.
        {"name": "prefill_chunk_512", "kind": "prefill_chunk", **gqa, "new": 512, "prefix": 32768},
        # One prompt of odd length through the C++ API at its default precision.
        {"name": "prefill_api_1500", "kind": "prefill_api", **gqa, "tokens": 1500},
        # FP32 caches (precision-critical use, and the original dtype of this API).
        {"name": "prefill_f32_4", "kind": "prefill_batch", **_shape("f32", 16, 4, 128, 16), "rows": 4, "lo": 384,
         "hi": 1024, "lens": 7},
        # A batch of forked requests (beam search, parallel sampling) that
        # all leave their shared tail pages.
        {"name": "cow_512", "kind": "cow", **gqa, "pairs": 512},
        # Idle requests' chunks to the CPU tier and back.
        {"name": "offload_256", "kind": "offload", "chunks": 256, "chunk_bytes": 65536},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["write", "gather", "decode", "decode", "decode", "decode_api", "prefill_batch",
                       "prefill_batch", "prefill_chunk", "prefill_api", "cow", "offload"])
    if kind == "offload":
        return {"kind": kind, "chunks": _log_int(rng, 8, 1024), "chunk_bytes": rng.choice([32768, 65536, 131072])}
    dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
    q_heads, kv_heads = rng.choice([(32, 8), (28, 4), (64, 8), (16, 4), (16, 2), (40, 8), (24, 8), (8, 8), (12, 1)])
    sizes = [64, 128, 128] if kind == "prefill_api" or dtype == "f32" else [64, 128, 128, 256]
    s = _shape(dtype, q_heads, kv_heads, rng.choice(sizes), rng.choice([8, 16, 16, 32, 64]))
    token = 2 * kv_heads * s["head_size"] * BYTES[dtype]  # K and V bytes of a token
    lens = rng.randrange(1 << 20)
    if kind == "write":
        return {"kind": kind, **s, "tokens": _log_int(rng, 1, 16384)}
    if kind == "cow":
        most = max(1, min(4096, int(2.5e8 / (token * s["block_size"]))))
        return {"kind": kind, **s, "pairs": _log_int(rng, 1, most)}
    if kind == "gather":
        rows = _log_int(rng, 1, 64)
        hi = _log_int(rng, 16, max(17, min(8192, int(1.0e9 / token / rows))))
        return {"kind": kind, **s, "rows": rows, "lo": max(1, hi // 16), "hi": hi, "lens": lens}
    if kind == "decode":
        rows = _log_int(rng, 1, 128)
        hi = _log_int(rng, 16, max(17, min(65536, int(5.0e9 / token / rows))))
        lo = max(1, hi // rng.choice([1, 2, 8, 32]))
        return {"kind": kind, **s, "rows": rows, "lo": lo, "hi": hi, "lens": lens,
                "prefix": rng.choice([0, 0, lo // 2]), "append": hi * rows * token < 3e8}
    if kind == "decode_api":
        rows = _log_int(rng, 1, 32)
        return {"kind": kind, **s, "rows": rows, "lo": 1, "hi": _log_int(rng, 16, 2048), "lens": lens}
    slow = 16 if dtype == "f32" else 1  # FP32 MFMAs run at a sixteenth of the rate
    if kind == "prefill_batch":
        rows = _log_int(rng, 1, 8)
        most = math.sqrt(8e11 / slow / (2 * q_heads * s["head_size"] * rows))
        hi = _log_int(rng, 16, max(17, min(4096, int(most))))
        return {"kind": kind, **s, "rows": rows, "lo": max(1, hi // rng.choice([1, 2, 8])), "hi": hi, "lens": lens}
    if kind == "prefill_chunk":
        new = _log_int(rng, 16, 2048)
        most = 6e11 / slow / (4 * q_heads * s["head_size"] * new)
        return {"kind": kind, **s, "new": new, "prefix": _log_int(rng, 16, max(17, min(65536, int(most))))}
    return {"kind": kind, **s, "tokens": _log_int(rng, 16, 2048)}


# ------------------------------------------------------------------ inputs
def _lengths(case):
    """The sequences' token counts (all of them at least `prefix` + 1)."""
    r = np.random.RandomState(case["lens"])
    n = r.randint(case["lo"], case["hi"] + 1, case["rows"])
    return np.maximum(n, case.get("prefix", 0) + 1).astype(np.int64)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, shape, dtype):
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _u64(values):
    """uint64 metadata on the GPU (as int64 tensors: the same bytes)."""
    return torch.as_tensor(np.ascontiguousarray(values).astype(np.int64), device="cuda")


def _tables(lengths, block_size, prefix, seed):
    """Random pages for every sequence: (table [rows][width], page count of
    the pool). The whole pages of the first `prefix` tokens are shared."""
    counts = -(-lengths // block_size)
    shared = prefix // block_size
    width = int(counts.max())
    own = counts - shared
    used = int(own.sum()) + shared
    pool = used + max(8, used // 16)  # a few pages belong to nobody
    order = np.random.RandomState(seed & 0x7fffffff).permutation(pool)
    table = np.full((len(lengths), width), -1, np.int64)
    table[:, :shared] = order[:shared]
    at = shared
    for r, n in enumerate(own):
        table[r, shared:shared + n] = order[at:at + n]
        at += n
    return table, pool


def _caches(case, pool, g):
    shape = (pool, case["kv_heads"], case["block_size"], case["head_size"])
    return _normal(g, shape, TORCH[case["dtype"]]), _normal(g, shape, TORCH[case["dtype"]])


def _sequences(case):
    """(lengths of the K/V, query tokens of each) of an attention case."""
    if case["kind"] == "prefill_chunk":
        return np.array([case["prefix"] + case["new"]]), np.array([case["new"]])
    if case["kind"] == "prefill_api":
        return np.array([case["tokens"]]), np.array([case["tokens"]])
    lengths = _lengths(case)
    if case["kind"] == "prefill_batch":
        return lengths, lengths
    return lengths, np.ones_like(lengths)


def _inputs(case, seed):
    """The inputs of a case as tensors, without any of this package's code."""
    g = _generator(seed)
    kind = case["kind"]
    if kind == "offload":
        return {"data": np.random.RandomState(seed & 0x7fffffff).randint(
            0, 256, (case["chunks"], case["chunk_bytes"]), np.uint8)}
    dt = TORCH[case["dtype"]]
    H, D, bs = case["kv_heads"], case["head_size"], case["block_size"]
    if kind == "cow":
        pool = 2 * case["pairs"] + max(8, case["pairs"] // 8)
        pairs = np.random.RandomState(seed & 0x7fffffff).permutation(pool)[:2 * case["pairs"]].reshape(-1, 2)
        k, v = _caches(case, pool, g)
        return {"k": k, "v": v, "pairs": pairs}
    if kind == "write":
        tokens = case["tokens"]
        table, pool = _tables(np.array([tokens]), bs, 0, seed)
        slots = table[0][np.arange(tokens) // bs] * bs + np.arange(tokens) % bs
        k, v = _caches(case, pool, g)
        return {"k": k, "v": v, "slots": slots, "new_k": _normal(g, (tokens, H, D), dt),
                "new_v": _normal(g, (tokens, H, D), dt)}
    if kind == "gather":
        lengths = _lengths(case)
        table, pool = _tables(lengths, bs, 0, seed)
        k, v = _caches(case, pool, g)
        return {"k": k, "v": v, "table": table, "lengths": lengths}
    lengths, queries = _sequences(case)
    q = _normal(g, (int(queries.sum()), case["q_heads"], D), torch.float32)
    if kind in ("decode_api", "prefill_api"):  # rows, written through the API
        total = int(lengths.sum())
        return {"rows_k": _normal(g, (total, H, D), dt), "rows_v": _normal(g, (total, H, D), dt), "q": q,
                "lengths": lengths, "queries": queries}
    table, pool = _tables(lengths, bs, case.get("prefix", 0) if kind == "decode" else 0, seed)
    k, v = _caches(case, pool, g)
    found = {"k": k, "v": v, "table": table, "lengths": lengths, "queries": queries, "q": q}
    if case.get("append"):
        found["new_k"] = _normal(g, (len(lengths), H, D), dt)
        found["new_v"] = _normal(g, (len(lengths), H, D), dt)
    return found


# ----------------------------------------------------------------- prepare
class _Bytes:
    """Memory that an object of this package owns, as an array interface; the
    views made from it keep the owner alive."""

    def __init__(self, owner, ptr, nbytes, device):
        self.owner = owner
        view = {"shape": (nbytes,), "typestr": "|u1", "data": (ptr, False), "version": 3}
        if device:
            self.__cuda_array_interface__ = {**view, "version": 2}
        else:
            self.__array_interface__ = view


def _prepare_offload(case, x):
    import kvflux_amd

    v2, v3 = kvflux_amd.v2, kvflux_amd.v3
    n, size = case["chunks"], case["chunk_bytes"]
    s = {"case": case, "pool": v2.PhysicalBlockPool(n, 16)}
    s["tiers"] = v3.GpuTier(s["pool"], size), v3.CpuTier(n, size), v3.NvmeTier(n, size)
    s["directory"] = v3.CacheDirectory(*s["tiers"])
    s["store"], s["host"] = v3.GpuChunkStore(n, size), v3.PinnedChunkPool(n, size)
    s["transfer"] = v3.GpuCpuTransfer(s["directory"], s["store"], s["host"])
    s["keys"] = [v3.make_cache_key("model", 1, v2.DType.BFloat16, 0, 32, [1, 2, 3, i]) for i in range(n)]
    for key, data in zip(s["keys"], x["data"]):
        s["directory"].create(key)
        slot = s["directory"].place(key, v3.StorageTier.CPU).slot
        C.memmove(s["host"].data(slot), data.ctypes.data, size)
    s["transfer"].begin_onload_batch(s["keys"])
    for key in s["keys"]:
        s["transfer"].finish_onload(key, True)
    gpu = min(s["store"].device_ptr(s["directory"].at(k).gpu.location) for k in s["keys"])
    host = min(s["host"].data(i) for i in range(n))
    s["gpu_bytes"] = torch.as_tensor(_Bytes(s["store"], gpu, n * size, True), device="cuda")
    s["host_bytes"] = np.asarray(_Bytes(s["host"], host, n * size, False))
    return s


def _prepare_api(case, x, seed):
    """Pool, storage and sequences of the C++ API, K/V written into random pages."""
    import kvflux_amd

    v2 = kvflux_amd.v2
    bs, lengths = case["block_size"], x["lengths"]
    pages = int((-(-lengths // bs)).sum())
    pool = v2.PhysicalBlockPool(pages + 8, bs)
    held = [pool.allocate() for _ in range(pages + 8)]
    for i in np.random.RandomState(seed & 0x7fffffff).permutation(pages + 8):
        pool.free(held[i])
    storage = v2.PagedKVStorage(pool, case["kv_heads"], case["head_size"], getattr(v2.DType, API_DTYPE[case["dtype"]]))
    sequences = []
    for r, n in enumerate(lengths):
        sequences.append(v2.SequenceState(r, pool))
        sequences[-1].append_tokens(int(n))
    slots = v2.build_slot_mapping([(s, t) for s in sequences for t in range(s.num_tokens())])
    torch.cuda.synchronize()
    v2.write_paged_kv(storage, x["rows_k"].data_ptr(), x["rows_v"].data_ptr(), slots)
    s = {"case": case, "v2": v2, "pool": pool, "storage": storage, "sequences": sequences, "q": x["q"],
         "out": torch.empty_like(x["q"])}
    if case["kind"] == "decode_api":
        s["table"] = v2.DeviceBatchTable(storage, sequences, int((-(-lengths // bs)).max()) + 1)
    return s


def prepare(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind == "offload":
        return _prepare_offload(case, x)
    if kind in ("decode_api", "prefill_api"):
        return _prepare_api(case, x, seed)
    from kvflux_amd import capi

    H, D, bs, Hq = case["kv_heads"], case["head_size"], case["block_size"], case["q_heads"]
    code = CODE[case["dtype"]]
    s = {"case": case, "capi": capi, "keep": x}
    cache = (x["k"].data_ptr(), x["v"].data_ptr(), x["k"].shape[0])
    if kind == "cow":
        s["pairs"] = _u64(x["pairs"])
        page = H * bs * D * BYTES[case["dtype"]]
        s["calls"] = [("kvflux_copy_pages", *cache, page, s["pairs"].data_ptr(), case["pairs"], None)]
        s["outputs"] = [x["k"], x["v"]]
        return s
    cache = (*cache, H, bs, D, code)
    if kind == "write":
        s["slots"] = _u64(x["slots"])
        s["calls"] = [("kvflux_write_paged_kv", *cache, x["new_k"].data_ptr(), x["new_v"].data_ptr(),
                       s["slots"].data_ptr(), case["tokens"], None)]
        s["outputs"] = [x["k"], x["v"]]
        return s
    lengths = x["lengths"]
    rows, width = x["table"].shape
    s["table"], s["lens"] = _u64(x["table"]), _u64(lengths)
    if kind == "gather":
        pages = -(-lengths // bs)
        s["offsets"] = _u64(np.cumsum(lengths) - lengths)
        s["starts"] = _u64(np.cumsum(pages) - pages)
        shape = (int(lengths.sum()), H, D)
        s["outputs"] = [torch.empty(shape, dtype=TORCH[case["dtype"]], device="cuda") for _ in range(2)]
        s["calls"] = [("kvflux_gather_paged_kv_live", *cache, s["table"].data_ptr(), width, s["lens"].data_ptr(),
                       s["offsets"].data_ptr(), s["starts"].data_ptr(), rows, int(pages.sum()),
                       s["outputs"][0].data_ptr(), s["outputs"][1].data_ptr(), None)]
        return s
    longest = int(lengths.max())
    out = torch.empty_like(x["q"])
    s["outputs"] = [out]
    size = C.c_size_t()
    if kind == "decode":
        s["calls"] = []
        if case["append"]:
            s["calls"].append(("kvflux_write_paged_kv_tail", *cache, x["new_k"].data_ptr(), x["new_v"].data_ptr(),
                               s["table"].data_ptr(), width, s["lens"].data_ptr(), rows, None))
            s["outputs"] += [x["k"], x["v"]]
        capi.call("kvflux_paged_attention_workspace_size", rows, longest, H, Hq, bs, D, C.byref(size))
        s["workspace"] = torch.empty(max(1, size.value), dtype=torch.uint8, device="cuda")
        s["calls"].append(("kvflux_paged_attention", *cache, s["table"].data_ptr(), width, s["lens"].data_ptr(),
                           longest, rows, Hq, x["q"].data_ptr(), out.data_ptr(), s["workspace"].data_ptr(),
                           size.value, None))
    elif kind == "prefill_batch":
        s["q_lens"] = _u64(x["queries"])
        s["q_offsets"] = _u64(np.cumsum(x["queries"]) - x["queries"])
        s["calls"] = [("kvflux_paged_prefill_batch", *cache, s["table"].data_ptr(), width, s["lens"].data_ptr(),
                       s["q_lens"].data_ptr(), s["q_offsets"].data_ptr(), rows, int(x["queries"].max()), longest, Hq,
                       x["q"].data_ptr(), out.data_ptr(), None)]
    else:
        capi.call("kvflux_paged_prefill_workspace_size", H, D, longest, case["new"], Hq, C.byref(size))
        s["workspace"] = torch.empty(max(1, size.value), dtype=torch.uint8, device="cuda")
        s["calls"] = [("kvflux_paged_prefill_split", *cache, s["table"].data_ptr(), width, longest, case["new"], Hq,
                       x["q"].data_ptr(), out.data_ptr(), s["workspace"].data_ptr(), size.value, None)]
    return s


# --------------------------------------------------------------------- run
def run(state):
    case = state["case"]
    if case["kind"] == "decode_api":
        state["v2"].paged_attention_batch(state["storage"], state["table"], state["q"].data_ptr(),
                                          state["out"].data_ptr(), case["q_heads"])
        return [state["out"]]
    if case["kind"] == "prefill_api":
        state["v2"].paged_attention(state["storage"], state["sequences"][0], state["q"].data_ptr(),
                                    state["out"].data_ptr(), case["tokens"], case["q_heads"])
        return [state["out"]]
    if case["kind"] == "offload":
        transfer, keys = state["transfer"], state["keys"]
        transfer.begin_offload_batch(keys)
        for key in keys:
            transfer.finish_offload(key, True)
        transfer.begin_onload_batch(keys)
        for key in keys:
            transfer.finish_onload(key, True)
        return [state["gpu_bytes"], state["host_bytes"]]
    call = state["capi"].call
    for name, *args in state["calls"]:
        call(name, *args)
    return state["outputs"]


# -------------------------------------------------------------------- work
def _visible(lengths, queries):
    """(query token, key) pairs of causal trailing queries."""
    return sum(int(q) * int(n - q) + int(q) * (int(q) + 1) // 2 for n, q in zip(lengths, queries))


def work(case):
    kind = case["kind"]
    if kind == "offload":
        return {"bytes": 4 * case["chunks"] * case["chunk_bytes"], "flops": 0}
    token = 2 * case["kv_heads"] * case["head_size"] * BYTES[case["dtype"]]
    if kind == "cow":
        return {"bytes": case["pairs"] * (2 * token * case["block_size"] + 16), "flops": 0}
    if kind == "write":
        return {"bytes": case["tokens"] * (2 * token + 8), "flops": 0}
    if kind == "gather":
        lengths = _lengths(case)
        return {"bytes": int(lengths.sum()) * 2 * token + 8 * int((-(-lengths // case["block_size"])).sum()),
                "flops": 0}
    lengths, queries = _sequences(case)
    shared = case.get("prefix", 0) // case["block_size"] * case["block_size"] if kind == "decode" else 0
    unique = int(lengths.sum()) - shared * (len(lengths) - 1)
    io = int(queries.sum()) * case["q_heads"] * case["head_size"] * 4 * 2
    table = 8 * int((-(-lengths // case["block_size"])).sum())
    more = 2 * token * len(lengths) if case.get("append") else 0
    return {"bytes": unique * token + io + table + more,
            "flops": 4 * case["q_heads"] * case["head_size"] * _visible(lengths, queries)}


# --------------------------------------------------------------- tolerance
def tolerance(case):
    kind = case["kind"]
    if kind in ("write", "gather", "cow", "offload"):
        return "exact"  # bytes are moved, none computed
    if kind in ("prefill_batch", "prefill_chunk") and case["dtype"] != "f32":
        # Q and the weights rounded to the cache's 16 bits: 2.4e-3 off the
        # 64-bit result in bf16, an eighth of that in f16.
        return {"rel": 9e-3, "max": 0.15} if case["dtype"] == "bf16" else {"rel": 1.2e-3, "max": 2e-2}
    return {"rel": 2e-6, "max": 4e-5}  # FP32 sums: 3e-7 off the 64-bit result


# ------------------------------------------------------------------- exact
def _attend(q, k, v, group):
    """q [T][Hq][D], k/v [L][H][D] in 64 bits; causal, the T last tokens query."""
    T, Hq, D = q.shape
    L = k.shape[0]
    out = torch.empty_like(q)
    past = L - T
    step = max(1, min(T, (1 << 27) // max(1, L * group)))  # about 1 GiB of scores
    for h in range(k.shape[1]):
        kh, vh = k[:, h, :].contiguous(), v[:, h, :].contiguous()
        kt = kh.t().contiguous()
        for a in range(0, T, step):
            b = min(T, a + step)
            seen = past + b
            qh = q[a:b, h * group:(h + 1) * group, :].reshape(-1, D).contiguous()
            w = (qh @ kt[:, :seen].contiguous()) / math.sqrt(D)
            if b - a > 1:
                at = past + a + torch.arange(b - a, device=q.device).repeat_interleave(group)
                w.masked_fill_(torch.arange(seen, device=q.device)[None, :] > at[:, None], float("-inf"))
            out[a:b, h * group:(h + 1) * group, :] = (torch.softmax(w, -1) @ vh[:seen]).reshape(b - a, group, D)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("write", "gather", "cow", "offload"):
        return None
    x = _inputs(case, seed)
    lengths, queries, bs = x["lengths"], x["queries"], case["block_size"]
    H, D = case["kv_heads"], case["head_size"]
    out = torch.empty(x["q"].shape, dtype=torch.float64, device="cuda")
    at = rows = 0
    for r, (n, t) in enumerate(zip(lengths, queries)):
        n, t = int(n), int(t)
        if "rows_k" in x:
            k, v = x["rows_k"][rows:rows + n].double(), x["rows_v"][rows:rows + n].double()
        else:
            pages = _u64(x["table"][r, :-(-n // bs)])
            k, v = (x[c][pages].permute(0, 2, 1, 3).reshape(-1, H, D)[:n].double() for c in ("k", "v"))
            if case.get("append"):
                k[n - 1], v[n - 1] = x["new_k"][r].double(), x["new_v"][r].double()
        out[at:at + t] = _attend(x["q"][at:at + t].double(), k, v, case["q_heads"] // H)
        at += t
        rows += n
    return [out] + ([None, None] if case.get("append") else [])
