"""The prefill attention's edges on the GPU: the row tiles (32 per wave, 128
per block), the 32-key tiles and the key ranges, against the float64 oracle
(rel 1e-4 on the floored metric, the attention tolerance); and values that the
kernel's three-term bf16 split does not cover (infinities, magnitudes whose
bf16 is infinite) or covers at the end of its range."""

from __future__ import annotations

import numpy as np
import pytest

from franken_ocr_amd import synth
from oracle import pyoracle as O

NH, D = 10, 128
DIM = NH * D

pytestmark = pytest.mark.gpu


def _run(ctx, q, k, v, c0):
    from franken_ocr_amd.engine import chunk_prefill_attention

    out = ctx.empty(q.shape, np.float32)
    chunk_prefill_attention(ctx.to_device(q), ctx.to_device(k), ctx.to_device(v), NH, D, c0, out)
    return out.numpy()


def _qkv(seed, rows, c0):
    n = rows + c0
    q = synth.f32_normal(synth.seed_of(seed), rows * DIM).reshape(rows, DIM)
    k, v = (synth.f32_normal(synth.seed_of(seed + i), n * DIM).reshape(n, DIM) for i in (1, 2))
    return q, k, v


def _close(got, want):
    want = np.asarray(want, np.float64)
    floor = np.abs(want).max(axis=-1, keepdims=True) * 1e-2
    err = np.abs(got.astype(np.float64) - want) / np.maximum(np.abs(want), floor)
    assert err.max() <= 1e-4, float(err.max())


@pytest.mark.parametrize("rows,c0", [(31, 0), (33, 1), (96, 31), (127, 33), (128, 0), (129, 640), (1, 2047), (260, 95),
                                     (192, 149), (193, 0), (64, 448), (64, 449), (1, 511), (1, 512), (66, 300)])
def test_row_and_key_tile_edges(ctx, rows, c0):
    q, k, v = _qkv(4100 + rows, rows, c0)
    st, want = O.chunk_prefill_attention(q, k, v, NH, D, c0)
    assert st == 0
    _close(_run(ctx, q, k, v, c0), want)


@pytest.mark.parametrize("scale", [1.0e34, 1.0e-34])
def test_values_at_the_ends_of_the_range(ctx, scale):
    # 1e-34 v: the split's third terms are subnormal. 1e34 v with two values
    # whose bf16 is infinite: the unnormalised sums (at most 3.399e38 + 330 *
    # 5e34 per value column) stay below f32's 3.403e38.
    q, k, v = _qkv(4300, 130, 200)
    v = (v * np.float32(scale)).astype(np.float32)
    if scale > 1:
        v[7, 5], v[150, 700] = 3.399e38, -3.399e38
    st, want = O.chunk_prefill_attention(q, k, v, NH, D, 200)
    assert st == 0 and np.isfinite(want).all()
    _close(_run(ctx, q, k, v, 200), want)


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_an_infinite_or_nan_value_reaches_the_rows_that_see_it(ctx, bad):
    rows, c0, key, col = 140, 70, 100, 3 * D + 9
    q, k, v = _qkv(4400, rows, c0)
    st, want = O.chunk_prefill_attention(q, k, v, NH, D, c0)
    v[key, col] = bad
    got = _run(ctx, q, k, v, c0)
    other = np.arange(DIM) != col
    _close(got[:, other], want[:, other])
    sees = np.arange(rows) + c0 >= key
    np.testing.assert_array_equal(got[sees, col], np.full(sees.sum(), bad, np.float32))


def test_a_key_of_minus_infinite_score_is_not_seen(ctx):
    rows, c0, key = 40, 60, 30
    q, k, v = _qkv(4500, rows, c0)
    q[:, :D] = np.abs(q[:, :D]) + 0.5
    k[key, 4] = -np.inf  # head 0's score of that key is -inf for every row
    k2, v2 = np.delete(k, key, 0), np.delete(v, key, 0)
    st, want = O.chunk_prefill_attention(q, k2, v2, NH, D, c0 - 1)
    assert st == 0
    _close(_run(ctx, q, k, v, c0)[:, :D], want[:, :D])
