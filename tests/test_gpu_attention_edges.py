"""The prefill attention's edges on the GPU: the row tiles (32 per wave, 128
per block), the 32-key tiles and the key ranges, against the float64 oracle
(rel 1e-4 on the floored metric, the attention tolerance); and values that the
large form's three-term bf16 split does not cover (infinities, magnitudes whose
bf16 is infinite) or covers at the end of its range. Up to 192 rows and 512
keys a call takes the small form, which has f32 products and no split: each of
these tests runs on both, 260 rows after 95 and 300 after 700 being past it."""

from __future__ import annotations

import ctypes

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


@pytest.mark.parametrize("rows,c0,scale", [(130, 200, 1.0e34), (130, 200, 1.0e-34), (260, 95, 1.0e31),
                                           (260, 95, 1.0e-34), (300, 700, 1.0e31), (300, 700, 1.0e-34)])
def test_values_at_the_ends_of_the_range(ctx, rows, c0, scale):
    # 1e-34 v: the split's third terms are subnormal. Large v with two values
    # whose bf16 is infinite: at 1e31 the unnormalised sums are at most
    # 3.399e38 + 1000 * 6e31, below f32's 3.403e38 (at 1e34 they are because
    # no row gives either value a probability near 1)
    q, k, v = _qkv(4300, rows, c0)
    v = (v * np.float32(scale)).astype(np.float32)
    if scale > 1:
        v[7, 5], v[150, 700] = 3.399e38, -3.399e38
    st, want = O.chunk_prefill_attention(q, k, v, NH, D, c0)
    assert st == 0 and np.isfinite(want).all()
    _close(_run(ctx, q, k, v, c0), want)


# three keys a tile apart: in ranges of two tiles or more, one of them at the
# least lies past its range's first tile
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("rows,c0,key", [(140, 70, 100), (260, 95, 100), (260, 95, 132), (260, 95, 164),
                                         (300, 700, 610), (300, 700, 642), (300, 700, 990)])
def test_an_infinite_or_nan_value_reaches_the_rows_that_see_it(ctx, rows, c0, key, bad):
    col = 3 * D + 9
    q, k, v = _qkv(4400, rows, c0)
    st, want = O.chunk_prefill_attention(q, k, v, NH, D, c0)
    v[key, col] = bad
    got = _run(ctx, q, k, v, c0)
    other = np.arange(DIM) != col
    _close(got[:, other], want[:, other])
    sees = np.arange(rows) + c0 >= key
    np.testing.assert_array_equal(got[sees, col], np.full(sees.sum(), bad, np.float32))


@pytest.mark.parametrize("rows,c0,key", [(40, 60, 30), (260, 95, 30), (260, 95, 62), (260, 95, 94), (300, 700, 610),
                                         (300, 700, 642)])
def test_a_key_of_minus_infinite_score_is_not_seen(ctx, rows, c0, key):
    q, k, v = _qkv(4500, rows, c0)
    q[:, :D] = np.abs(q[:, :D]) + 0.5
    k[key, 4] = -np.inf  # head 0's score of that key is -inf for every row
    k2, v2 = np.delete(k, key, 0), np.delete(v, key, 0)
    st, want = O.chunk_prefill_attention(q, k2, v2, NH, D, c0 - 1)
    assert st == 0
    _close(_run(ctx, q, k, v, c0)[:, :D], want[:, :D])


@pytest.mark.parametrize("rows,c0", [(40, 60), (260, 95), (300, 700)])
def test_a_finite_key_whose_bf16_is_infinite(ctx, rows, c0):
    q, k, v = _qkv(4600, rows, c0)
    q[:, 4] = 0.0  # head 0 does not look at the dim
    st, want = O.chunk_prefill_attention(q, k, v, NH, D, c0)
    assert st == 0
    k[c0 + 20, 4], k[5, 4] = 3.399e38, -3.399e38
    _close(_run(ctx, q, k, v, c0), want)


@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("rows,c0", [(40, 60), (260, 95), (300, 700)])
def test_a_query_that_is_not_finite_stays_in_its_row(ctx, rows, c0, bad):
    q, k, v = _qkv(4700, rows, c0)
    st, want = O.chunk_prefill_attention(q, k, v, NH, D, c0)
    assert st == 0
    row = rows - 7
    q[row, D + 3] = bad  # head 1
    got = _run(ctx, q, k, v, c0)
    assert np.isnan(got[row, D:2 * D]).all()
    keep = np.ones_like(got, bool)
    keep[row, D:2 * D] = False
    want = np.where(keep, want, 0.0)
    _close(np.where(keep, got, 0.0), want)


@pytest.mark.parametrize("rows,c0", [(40, 60), (260, 95), (300, 700)])
@pytest.mark.parametrize("sq,sk,sv", [(1.0, 1.0, 1e-35), (1.0, 1.0, 1e-37), (1e-36, 1e36, 1.0), (1e36, 1e-36, 1.0)])
def test_values_too_small_for_three_bf16_terms(ctx, rows, c0, sq, sk, sv):
    """Magnitudes whose third bf16 term has no bits left (f32 products keep
    them, subnormal results included), among zeros, which have a split."""
    q, k, v = _qkv(4800, rows, c0)
    q, k, v = (q * np.float32(sq)).astype(np.float32), (k * np.float32(sk)).astype(np.float32), v * np.float32(sv)
    v[::3] = 0.0
    k[1::3] = 0.0
    st, want = O.chunk_prefill_attention(q, k, v, NH, D, c0)
    assert st == 0
    _close(_run(ctx, q, k, v, c0), want)


def _f32_rows(q, k, v, c0):
    """The attention in f32 scores: for scores so large that f32 decides which
    key is the row's largest, the f64 softmax of the f32 scores."""
    out = np.empty(q.shape, np.float64)
    for h in range(NH):
        cols = slice(h * D, (h + 1) * D)
        for i in range(q.shape[0]):
            s = (k[:c0 + i + 1, cols].astype(np.float64) @ q[i, cols].astype(np.float64)).astype(np.float32)
            s = s.astype(np.float64) / np.sqrt(D)
            p = np.exp(s - s.max())
            out[i, cols] = p @ v[:c0 + i + 1, cols].astype(np.float64) / p.sum()
    return out


@pytest.mark.parametrize("rows,c0", [(40, 60), (260, 95)])
@pytest.mark.parametrize("scale", [1e5, 1e12, 1e18])
def test_scores_far_from_zero(ctx, rows, c0, scale):
    """q and k of about that size: one key has all of a row's probability, and
    the outputs are its value, whatever the scores' ulp (1e5: of 2^13, 1e12: of
    2^59). A key is close enough to a row's largest to share it in none of them
    (their gaps are some 1e-4 of the scores at the least)."""
    q, k, v = _qkv(4900, rows, c0)
    q, k = q * np.float32(scale), k * np.float32(scale)
    _close(_run(ctx, q, k, v, c0), _f32_rows(q, k, v, c0))


@pytest.mark.parametrize("rows,c0", [(40, 60), (260, 95), (300, 700)])
def test_scores_that_overflow_downwards(ctx, rows, c0):
    """Keys whose score is below f32's range have no probability; a row's other
    keys are attended as ever (the last 20 columns of every 64 keys are such)."""
    q, k, v = _qkv(5000, rows, c0)
    low = np.arange(rows + c0) % 64 >= 44
    q[:, 4::D] = 1e21
    k[:, 4::D] = 0.0
    less = k.copy()
    less[low, 4::D] = -1e10  # as little probability, within range
    st, want = O.chunk_prefill_attention(q, less, v, NH, D, c0)
    assert st == 0 and np.isfinite(want).all()
    k[low, 4::D] = -1e21 * synth.f32_uniform(synth.seed_of(5003), low.sum() * NH, 1.0, 1.02).reshape(-1, NH)
    _close(_run(ctx, q, k, v, c0), want)


@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("rows,c0", [(64, 440), (260, 95), (300, 700)])
def test_a_value_that_is_not_finite_shows_at_probability_zero(ctx, rows, c0, bad):
    """A key so far below the rows' largest score that its probability is 0 in
    f32: 0 * inf and 0 * NaN are NaN, also where its whole key range (key 0's:
    every key but the last 40) is that far below."""
    q, k, v = _qkv(5100, rows, c0)
    q[:, 4::D], k[:, 4::D] = 40.0, 0.0
    k[c0 - 40:c0, 4::D] = 60.0  # + 212 in these keys' scores
    v[0, 5] = bad
    got = _run(ctx, q, k, v, c0)
    assert np.isnan(got[:, 5]).all()
    assert np.isfinite(np.delete(got, 5, 1)).all()


def test_a_long_call_keeps_its_partials_within_bounds(ctx):
    """32768 rows over 32768 keys: the key ranges' partials stay within 512 MiB
    of scratch (ranges as short as the time alone asks for would take 3.2 GB),
    and the rows are right."""
    from franken_ocr_amd.engine import chunk_prefill_attention

    rows = 32768
    path = next(ln.split()[-1] for ln in open("/proc/self/maps") if "libamdhip64" in ln)
    hip, free, total = ctypes.CDLL(path), ctypes.c_size_t(), ctypes.c_size_t()
    x = np.tile(synth.f32_normal(synth.seed_of(5200), 512 * DIM).reshape(512, DIM), (rows // 512, 1))
    dx, out = ctx.to_device(x), ctx.empty((rows, DIM), np.float32)
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    before = free.value
    chunk_prefill_attention(dx, dx, dx, NH, D, 0, out)
    got = out.numpy()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    assert before - free.value <= (512 << 20) + (64 << 20), before - free.value
    for row in (0, 4097, 20000, rows - 1):
        keys = x[:row + 1].reshape(-1, NH, D)
        s = np.einsum("khd,hd->hk", keys, x[row].reshape(NH, D), dtype=np.float64) / np.sqrt(D)
        p = np.exp(s - s.max(axis=1, keepdims=True))
        p /= p.sum(axis=1, keepdims=True)
        _close(got[row], np.einsum("hk,khd->hd", p, keys, dtype=np.float64).reshape(-1))


@pytest.mark.parametrize("rows,c0", [(40, 60), (130, 382), (260, 95), (300, 700)])
def test_rows_that_start_anywhere(ctx, rows, c0):
    """q, k, v and the output four bytes past a 16-byte boundary: the same bits."""
    from franken_ocr_amd.engine import chunk_prefill_attention

    q, k, v = _qkv(5300, rows, c0)

    def view(a):
        buf = ctx.to_device(np.concatenate([np.zeros(1, np.float32), a.reshape(-1)]).reshape(-1, 1))
        part = buf.view_rows(1, 1 + a.size)
        part.shape = a.shape
        assert part.ptr % 16 == 4
        return part

    out = view(np.zeros_like(q))
    chunk_prefill_attention(view(q), view(k), view(v), NH, D, c0, out)
    np.testing.assert_array_equal(out.numpy(), _run(ctx, q, k, v, c0))
