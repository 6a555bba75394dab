"""FP32-cache prefill over FP32's whole range: values that three BF16 parts
cannot stand for, or whose part products leave the range where the FP32
product of the whole values does not, are computed on FP32 MFMAs. Against the
oracle, relative to the size of the outputs.
"""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import DTYPES, buffer_like
from kvflux_amd import capi, device
from oracle import oracle
from test_gpu_prefill_parts import arena

pytestmark = pytest.mark.gpu

SHAPES = [(128, 16, 200, 200), (64, 4, 300, 40)]  # head size, block size, kv tokens, query tokens


def prefill(kc, vc, blocks, kv_heads, bs, D, td, width, kv, tq, q_heads, q):
    qd, out = buffer_like(q.reshape(-1)), buffer_like(np.full(q.size, 7.0, np.float32))
    capi.check(capi.lib().kvflux_paged_prefill(kc.ptr, vc.ptr, blocks, kv_heads, bs, D, DTYPES["Float32"][0], td.ptr,
                                               width, kv, tq, q_heads, qd.ptr, out.ptr, None))
    device.synchronize()
    return out.download(np.float32).reshape(tq, q_heads, D)


def run(D, bs, kv, tq, seed, change):
    """(outputs, oracle) after change(keys, values, queries), each [token][head][dim]."""
    kv_heads, q_heads = 2, 8
    code, host = DTYPES["Float32"]
    kc, vc, blocks, table, width = arena("Float32", kv_heads, bs, D, [kv], seed)
    kh, vh = kc.download(host).reshape(blocks, kv_heads, bs, D), vc.download(host).reshape(blocks, kv_heads, bs, D)
    q = oracle.random_elements(0, tq * q_heads * D, oracle.F32, 1, seed + 2).reshape(tq, q_heads, D)
    pages, rows = table[0, np.arange(kv) // bs].astype(np.int64), np.arange(kv) % bs
    k, v = kh[pages, :, rows], vh[pages, :, rows]
    change(k, v, q)
    kh[pages, :, rows], vh[pages, :, rows] = k, v
    kc.upload(kh.reshape(-1))
    vc.upload(vh.reshape(-1))
    exp = oracle.paged_attention_causal(kh.reshape(-1), vh.reshape(-1), kv_heads, bs, D, code, table[0], kv,
                                        q.reshape(-1), tq, q_heads, threads=8).reshape(tq, q_heads, D)
    return prefill(kc, vc, blocks, kv_heads, bs, D, buffer_like(table.reshape(-1)), width, kv, tq, q_heads, q), exp


def bf16(x):
    """x rounded to the nearest BF16 value (finite x)."""
    bits = np.asarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return ((bits + 0x7fff + ((bits >> np.uint64(16)) & np.uint64(1))) & np.uint64(0xffff0000)).astype(np.uint32).view(
        np.float32)


@pytest.mark.parametrize("D,bs,kv,tq", SHAPES)
@pytest.mark.parametrize("element", [-1.003e38, -1.005e38])
def test_finite_elements_whose_score_overflows(gpu, D, bs, kv, tq, element):
    """A key whose score is below the lowest FP32 value is dropped (weight 0),
    whatever the sign of the element's second part."""
    mid = float(np.float32(element)) - float(bf16(element))
    assert (mid > 0) == (element == -1.003e38)

    def change(k, v, q):
        k[:, :, 3] = 0.0
        k[(kv - tq) // 2 + 1, :, 3] = element
        q[:, :, 3] = 2e4 * np.sqrt(D) / 1.4427  # 2e4 once scaled

    got, exp = run(D, bs, kv, tq, 1000 + kv, change)
    assert np.all(np.isfinite(got))
    assert np.abs(got - exp).max() < 1e-5


@pytest.mark.parametrize("D,bs,kv,tq", SHAPES)
@pytest.mark.parametrize("power", [-100, -110, -120])
def test_small_values(gpu, D, bs, kv, tq, power):
    """V near 2^power: relative to it, the outputs are those of V near 1."""
    got, exp = run(D, bs, kv, tq, 1020 + kv, lambda k, v, q: np.ldexp(v, power, out=v))
    assert np.abs(got.astype(np.float64) - exp).max() < 1e-6 * 2.0 ** power * 4


@pytest.mark.parametrize("D,bs,kv,tq", SHAPES)
@pytest.mark.parametrize("power", [100, 118])
def test_small_keys_large_queries(gpu, D, bs, kv, tq, power):
    """K near 2^-power and Q near 2^power: the scores of both near 1."""
    def change(k, v, q):
        np.ldexp(k, -power, out=k)
        np.ldexp(q, power, out=q)

    got, exp = run(D, bs, kv, tq, 1040 + kv, change)
    assert np.abs(got - exp).max() < 1e-5


@pytest.mark.parametrize("D,bs,kv,tq", SHAPES)
def test_small_weights(gpu, D, bs, kv, tq):
    """A column whose only nonzero V belongs to a key of weight near 2^-121:
    its outputs are that weight's. The queries have one nonzero dimension, so
    its score is one product (later dimensions add exact zeros): at most four
    roundings of values up to 128, 2^-18 each, and the query's and the scale's
    own, 2^-24 of 121 each: (2^-16 + 242 * 2^-24) * ln 2 = 2.1e-5 of the weight."""
    key = (kv - tq) // 2 + 2

    def change(k, v, q):
        k[:, :, 3] = 0.0
        q[:] = 0.0
        q[:, :, 3] = 8.0
        k[key, :, 3] = -120.5 / 8.0 * np.sqrt(D) / 1.4427
        v[:, :, 7] = 0.0
        v[key, :, 7] = 1.2345678 * 2.0 ** 20

    got, exp = run(D, bs, kv, tq, 1060 + kv, change)
    rows = slice(max(0, key + 1 - (kv - tq)), None)
    assert np.abs(exp[rows, :, 7]).min() > 2.0 ** -126
    assert np.abs(got[rows, :, 7] / exp[rows, :, 7].astype(np.float64) - 1).max() < 3e-5
    assert np.abs(got - exp).max() < 1e-5


@pytest.mark.parametrize("D,bs,kv,tq", SHAPES)
def test_mantissas_that_lose_most(gpu, D, bs, kv, tq):
    """K, Q and V of the mantissa whose part products left out weigh most
    (2^-24 of a product) at random signs and powers of two: the scores move by
    at most 2^-24 * sum |q k| / sqrt(D) <= 2^-24 sqrt(D) * 2.3, the outputs by
    that and a rounding of each: under 2e-6, the sums' own roundings aside."""
    rng = np.random.default_rng(kv)

    def change(k, v, q):
        for x in (k, v, q):
            x[:] = rng.choice([-1.0, 1.0], x.shape) * np.float32(1.0038986) * np.exp2(-rng.integers(0, 3, x.shape))

    got, exp = run(D, bs, kv, tq, 1080 + kv, change)
    assert np.abs(got - exp).max() < 1e-5
    assert np.sqrt(((got - exp).astype(np.float64) ** 2).mean()) < 1e-6
