"""Prefill launches whose wavefronts split the keys of a workgroup (small
grids, 16-bit caches): rows whose only keys lie in one half of a tile, last
tiles with one or both halves live, groups at and past the halved row count,
every head size, key splits beside them, and rows without a finite score. Every
case names the plan that it is there for and asserts it. The FP32 kernel, which
has no key parts, runs the same shapes. FP32 caches and the exact path at 1e-5
against the oracle over whole outputs, the rounded path at 2e-2.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from gpu_util import DTYPES, buffer_like
from kvflux_amd import capi, device
from oracle import oracle

pytestmark = pytest.mark.gpu


def arena(name, kv_heads, bs, head_size, kv_lens, seed):
    """Random pages for every sequence: (k, v, pages, table, width)."""
    code, host = DTYPES[name]
    width = max(-(-int(n) // bs) for n in kv_lens) + 1
    blocks = len(kv_lens) * width + 2
    page = kv_heads * bs * head_size
    kc = device.DeviceBuffer(blocks * page * np.dtype(host).itemsize)
    vc = device.DeviceBuffer(blocks * page * np.dtype(host).itemsize)
    device.fill_random(kc.ptr, blocks * page, code, 1, seed)
    device.fill_random(vc.ptr, blocks * page, code, 1, seed + 1)
    order = np.random.default_rng(seed).permutation(blocks).astype(np.uint64)
    table = np.full((len(kv_lens), width), 2**64 - 1, np.uint64)
    for i, n in enumerate(kv_lens):
        pages = -(-int(n) // bs)
        table[i, :pages] = order[i * width:i * width + pages]
    return kc, vc, blocks, table, width


def plan(name, kv_heads, q_heads, head_size, kv, tq, exact=False, workspace=False):
    """(key splits, key parts) that the call launches."""
    splits, parts = C.c_uint32(0), C.c_uint32(0)
    capi.check(capi.lib().kvflux_paged_prefill_plan(kv_heads, head_size, DTYPES[name][0], int(exact), kv, tq, q_heads,
                                                    int(workspace), C.byref(splits), C.byref(parts)))
    return splits.value, parts.value


SHAPES = [  # name, kv heads, q heads, D, block size, (kv, queries) of each sequence
    ("BFloat16", 2, 8, 128, 16, [(1, 1), (31, 31), (33, 33), (64, 64), (65, 65)]),
    ("Float16", 1, 4, 128, 8, [(97, 97), (320, 1), (352, 40), (130, 130)]),  # rows starting in either half
    ("BFloat16", 1, 128, 128, 16, [(70, 70)]),   # a group of exactly half the rows (one token a workgroup)
    ("BFloat16", 1, 129, 128, 16, [(70, 70)]),   # one past it: one key part
    ("Float16", 2, 6, 64, 1, [(200, 200), (63, 5)]),
    ("BFloat16", 1, 3, 256, 32, [(129, 129), (512, 33)]),
    ("Float32", 2, 8, 128, 16, [(1, 1), (32, 32), (33, 33), (300, 300), (161, 7)]),
    ("Float32", 1, 64, 64, 16, [(96, 96)]),
    ("Float32", 1, 65, 64, 4, [(96, 96)]),
]


@pytest.mark.parametrize("case", range(len(SHAPES)))
def test_key_parts(gpu, case):
    name, kv_heads, q_heads, D, bs, seqs = SHAPES[case]
    code, host = DTYPES[name]
    kv = np.array([a for a, _ in seqs], np.uint64)
    ql = np.array([b for _, b in seqs], np.uint64)
    for a, b in seqs:
        assert plan(name, kv_heads, q_heads, D, a, b) == (1, 1 if name == "Float32" or q_heads == 129 else 2)
    off = np.concatenate([[0], np.cumsum(ql)[:-1]]).astype(np.uint64)
    kc, vc, blocks, table, width = arena(name, kv_heads, bs, D, kv, 700 + 2 * case)
    total, row = int(ql.sum()), q_heads * D
    q = oracle.random_elements(0, total * row, oracle.F32, 1, 750 + case)
    td, qd = buffer_like(table.reshape(-1)), buffer_like(q)
    out = buffer_like(np.full(total * row + 8, 7.0, np.float32))
    for i in range(len(seqs)):
        at = int(off[i]) * row * 4
        capi.check(capi.lib().kvflux_paged_prefill_split(kc.ptr, vc.ptr, blocks, kv_heads, bs, D, code,
                                                         td.ptr + i * width * 8, width, int(kv[i]), int(ql[i]),
                                                         q_heads, qd.ptr + at, out.ptr + at, None, 0, None))
    device.synchronize()
    got = out.download(np.float32)
    assert np.all(got[total * row:] == 7.0)
    got = got[:total * row]
    rows = np.concatenate([np.full(b, i) for i, (_, b) in enumerate(seqs)])
    lens = np.concatenate([np.arange(a - b + 1, a + 1) for a, b in seqs]).astype(np.uint64)
    exp = oracle.paged_attention_rows(kc.download(host), vc.download(host), kv_heads, bs, D, code,
                                      table[rows].reshape(-1), width, lens, q, q_heads, threads=8)
    assert np.all(np.isfinite(got))
    assert np.abs(got - exp).max() < (1e-5 if name == "Float32" else 2e-2)


SINGLE = [  # exact, name, kv heads, q heads, D, block size, kv, query tokens, plans with and without a workspace
    (True, "BFloat16", 2, 8, 128, 16, 33, 33, (1, 1), (1, 1)),
    (True, "BFloat16", 2, 8, 128, 16, 1500, 20, (6, 2), (1, 2)),     # key splits beside the parts
    (True, "Float16", 4, 28, 128, 16, 257, 257, (1, 2), (1, 2)),
    (True, "Float16", 1, 2, 64, 32, 1000, 16, (4, 1), (1, 2)),
    (True, "Float32", 4, 16, 128, 16, 2000, 128, (8, 1), (1, 1)),
    (True, "BFloat16", 1, 4, 64, 8, 640, 640, (2, 1), (1, 2)),
    (False, "BFloat16", 2, 8, 128, 16, 1500, 20, (6, 2), (1, 2)),
    (False, "Float16", 8, 32, 128, 16, 4096, 64, (13, 2), (1, 2)),
    (False, "BFloat16", 1, 4, 64, 8, 1000, 33, (4, 2), (1, 2)),
    (False, "Float16", 2, 8, 256, 32, 600, 40, (2, 2), (1, 2)),
    (False, "BFloat16", 8, 32, 256, 16, 3000, 200, (4, 1), (1, 2)),
]


@pytest.mark.parametrize("case", range(len(SINGLE)))
def test_key_parts_and_splits(gpu, case):
    exact, name, kv_heads, q_heads, D, bs, kv, tq, with_splits, without = SINGLE[case]
    assert plan(name, kv_heads, q_heads, D, kv, tq, exact, True) == with_splits
    assert plan(name, kv_heads, q_heads, D, kv, tq, exact, False) == without
    code, host = DTYPES[name]
    kc, vc, blocks, table, width = arena(name, kv_heads, bs, D, [kv], 800 + 2 * case)
    q = oracle.random_elements(0, tq * q_heads * D, oracle.F32, 1, 850 + case)
    need = C.c_size_t(0)
    capi.check(capi.lib().kvflux_paged_prefill_workspace_size(kv_heads, D, kv, tq, q_heads, C.byref(need)))
    exp = oracle.paged_attention_causal(kc.download(host), vc.download(host), kv_heads, bs, D, code, table[0], kv, q,
                                        tq, q_heads, threads=8)
    td, qd = buffer_like(table.reshape(-1)), buffer_like(q)
    entry = getattr(capi.lib(), "kvflux_paged_prefill_exact" if exact else "kvflux_paged_prefill_split")
    for size in (need.value, 0):  # with and without room for key splits
        ws = buffer_like(np.full(size // 4 + 8, np.nan, np.float32))
        out = buffer_like(np.full(q.size + 8, 7.0, np.float32))
        capi.check(entry(kc.ptr, vc.ptr, blocks, kv_heads, bs, D, code, td.ptr, width, kv, tq, q_heads, qd.ptr,
                         out.ptr, ws.ptr if size else None, size, None))
        device.synchronize()
        got = out.download(np.float32)
        assert np.all(got[q.size:] == 7.0) and np.all(np.isnan(ws.download(np.float32)[size // 4:]))
        assert np.abs(got[:q.size] - exp).max() < (1e-5 if exact else 2e-2)


@pytest.mark.parametrize("name,D,exact,kv", [
    ("BFloat16", 64, False, 150), ("BFloat16", 128, False, 150), ("BFloat16", 256, False, 150),
    ("Float16", 128, False, 150), ("BFloat16", 64, True, 640), ("BFloat16", 128, True, 200),
])
def test_rows_without_a_score_above_minus_infinity(gpu, name, D, exact, kv):
    """Two key parts: the first keys score -inf for every row (their products
    overflow; FP16: an infinite element), so the rows that see no other key
    have no softmax and come out NaN, as with one key part; a key with a NaN
    makes every row that sees it NaN; the rows between are the oracle's."""
    kv_heads, q_heads, bs, none, nan = 2, 8, 16, 6, 70
    assert plan(name, kv_heads, q_heads, D, kv, kv, exact) == (1, 2)
    code, host = DTYPES[name]
    kc, vc, blocks, table, width = arena(name, kv_heads, bs, D, [kv], 870 + D)
    kh = kc.download(host).reshape(blocks, kv_heads, bs, D)
    at = lambda t: (int(table[0, t // bs]), slice(None), t % bs)  # noqa: E731
    for t in range(none):
        kh[at(t)][:, 3] = 0x7c00 if name == "Float16" else 0x7f62  # inf, 3.004e38
    q = oracle.random_elements(0, kv * q_heads * D, oracle.F32, 1, 890).reshape(kv, q_heads, D)
    q[:, :, 3] = -40.0
    exp = oracle.paged_attention_causal(kh.reshape(-1), vc.download(host), kv_heads, bs, D, code, table[0], kv,
                                        q.reshape(-1), kv, q_heads, threads=8).reshape(kv, q_heads, D)
    kh[at(nan)][:, 9] = 0x7fff
    kc.upload(kh.reshape(-1))
    td, qd = buffer_like(table.reshape(-1)), buffer_like(q.reshape(-1))
    args = (kc.ptr, vc.ptr, blocks, kv_heads, bs, D, code, td.ptr, width, kv, kv, q_heads, qd.ptr)
    out = buffer_like(np.full(q.size, 7.0, np.float32))
    capi.check(getattr(capi.lib(), "kvflux_paged_prefill_exact" if exact else "kvflux_paged_prefill_split")(
        *args, out.ptr, None, 0, None))
    device.synchronize()
    got = out.download(np.float32).reshape(kv, q_heads, D)
    assert np.all(np.isnan(got[:none])) and np.all(np.isnan(got[nan:]))
    assert np.abs(got[none:nan] - exp[none:nan]).max() < (1e-5 if exact else 2e-2)
    if not exact:  # the entry without key parts
        capi.check(capi.lib().kvflux_paged_prefill(*args, out.ptr, None))
        device.synchronize()
        assert np.array_equal(np.isnan(out.download(np.float32)), np.isnan(got.reshape(-1)))


@pytest.mark.parametrize("D,exact", [(64, False), (128, False), (256, False), (128, True)])
def test_missing_page_in_two_key_parts(gpu, D, exact):
    """A table entry outside the pool in the middle of the sequence: its keys
    and values read as zeros, as with one key part."""
    name, kv_heads, q_heads, bs, kv = "BFloat16", 2, 8, 16, 150
    assert plan(name, kv_heads, q_heads, D, kv, kv, exact) == (1, 2)
    code, host = DTYPES[name]
    kc, vc, blocks, table, width = arena(name, kv_heads, bs, D, [kv], 920 + D)
    kh, vh = (x.download(host).reshape(blocks, -1) for x in (kc, vc))
    spare = next(b for b in range(blocks) if b not in set(table[0].tolist()))
    kh[spare] = vh[spare] = 0
    q = oracle.random_elements(0, kv * q_heads * D, oracle.F32, 1, 940)
    for page in (1, 2, 5):  # in the first, the second half of a tile
        known, asked = table.copy(), table.copy()
        known[0, page], asked[0, page] = spare, 2**64 - 1 - page
        exp = oracle.paged_attention_causal(kh.reshape(-1), vh.reshape(-1), kv_heads, bs, D, code, known[0], kv, q, kv,
                                            q_heads, threads=8)
        td, qd, out = buffer_like(asked.reshape(-1)), buffer_like(q), buffer_like(np.full(q.size, 7.0, np.float32))
        capi.check(getattr(capi.lib(), "kvflux_paged_prefill_exact" if exact else "kvflux_paged_prefill_split")(
            kc.ptr, vc.ptr, blocks, kv_heads, bs, D, code, td.ptr, width, kv, kv, q_heads, qd.ptr, out.ptr, None, 0,
            None))
        device.synchronize()
        assert np.abs(out.download(np.float32) - exp).max() < (1e-5 if exact else 2e-2)


@pytest.mark.parametrize("D,bs,kv,tq", [(128, 16, 200, 200), (64, 1, 2500, 40), (128, 4, 9000, 33)])
def test_f32_values_without_parts(gpu, D, bs, kv, tq):
    """FP32 caches enter BF16 MFMAs as three parts each; infinities and values
    that round to one in BF16 have none. A key with an infinite element that
    every row scores -inf drops out, V keeps values near the largest float,
    and an infinite query element (first row) leaves the other rows alone."""
    kv_heads, q_heads = 2, 8
    code, host = DTYPES["Float32"]
    kc, vc, blocks, table, width = arena("Float32", kv_heads, bs, D, [kv], 900 + kv)
    kh, vh = kc.download(host).reshape(blocks, kv_heads, bs, D), vc.download(host).reshape(blocks, kv_heads, bs, D)
    q = oracle.random_elements(0, tq * q_heads * D, oracle.F32, 1, 950).reshape(tq, q_heads, D)
    q[:, :, 3] = -np.abs(q[:, :, 3]) - 3
    at = lambda t: (int(table[0, t // bs]), slice(None), t % bs)  # noqa: E731
    seen = kv - tq  # every row sees the keys up to here
    # Not key 0: with tq == kv it is the first row's only key, and a row whose
    # every score is -inf has no softmax.
    dropped, big = seen // 2 + 1, max(seen - 40, 2)
    kh[at(dropped)][:, 3] = np.inf
    # Weights are relative to a reference point up to 2^8 below the largest
    # score, so a key of ordinary score would overflow the sum itself: this one
    # scores 3 * 30 / sqrt(D) (8 or more) below the others.
    kh[at(big)][:, 3] = 30.0
    vh[at(big)][:, 5] = 3.4e38
    kc.upload(kh.reshape(-1))
    vc.upload(vh.reshape(-1))
    exp = oracle.paged_attention_causal(kh.reshape(-1), vh.reshape(-1), kv_heads, bs, D, code, table[0], kv,
                                        q.reshape(-1), tq, q_heads, threads=8).reshape(tq, q_heads, D)
    td = buffer_like(table.reshape(-1))
    for bad_row in (False, True):
        if bad_row:
            q[0, 0, 7] = np.inf
        qd, out = buffer_like(q.reshape(-1)), buffer_like(np.full(q.size, 7.0, np.float32))
        capi.check(capi.lib().kvflux_paged_prefill(kc.ptr, vc.ptr, blocks, kv_heads, bs, D, code, td.ptr, width, kv,
                                                   tq, q_heads, qd.ptr, out.ptr, None))
        device.synchronize()
        got = out.download(np.float32).reshape(tq, q_heads, D)
        rest = np.ones((tq, q_heads), bool)
        rest[0, 0] = not bad_row
        # Rows that see the key dropped or the large value: relative there.
        assert np.all(np.isfinite(got[rest]))
        err = np.abs(got.astype(np.float64) - exp) / np.maximum(1.0, np.abs(exp))
        # Column 5 is the large value times one weight, whose relative error
        # is ln 2 times its score's: scores down to -64 (log2) round at 2^-19
        # in each of the kernel's up to 32 steps, 32 * 2^-19 * ln 2 = 4.3e-5.
        assert np.delete(err, 5, axis=2)[rest].max() < 1e-5
        assert err[rest][:, 5].max() < 5e-5
