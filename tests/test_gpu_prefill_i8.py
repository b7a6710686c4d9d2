"""GPU parity for the prefill path on int8 weights (int8 matrix cores, i32
accumulation): nn::linear_int8_dynamic (nn.rs:151-173) and moe_block_i8
(decoder.rs:2142-2181) against the CPU oracle.

The linear's outputs are bit-exact: the activation bytes follow the same
rule (true division, ties to even), the i32 sums are exact, and the dequant
is the same two rounded multiplies (+ bias). The MoE block is compared within
rel 1e-3 (the MoE configs' layer-output tolerance): SiLU goes
through expf, which may differ from glibc's by an ulp and flip an act code
in the re-quantization, everything else is the same arithmetic."""

from __future__ import annotations

import numpy as np
import pytest

from franken_ocr_amd import synth
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

H, I, E, K = 1280, 896, 64, 6


def _say(msg):
    print(f"[gpu-prefill-i8] {msg}", flush=True)


def assert_rel(got, want, rtol):
    want = np.asarray(want, np.float64)
    scale = np.maximum(np.abs(want), np.abs(want).max() * 1e-2)
    rel = np.abs(np.asarray(got, np.float64) - want) / scale
    assert rel.max() <= rtol, f"max rel err {rel.max():.3e} > {rtol}"


@pytest.mark.parametrize("m,k,n,bias", [(1, 64, 8, False), (5, 128, 33, True), (64, 1280, 256, False),
                                        (100, 1280, 3840, True), (513, 896, 1280, False), (7, 6848, 64, True),
                                        (130, 1792, 300, False), (256, 1280, 256, True), (700, 960, 1000, True),
                                        (300, 6848, 96, False), (512, 1280, 6848, True), (257, 192, 33, True),
                                        (256, 8256, 40, True), (256, 1280, 1280, False), (17, 1280, 3840, False),
                                        (200, 6848, 1280, False), (256, 1792, 1280, False)])
def test_linear_i8_dynamic_bit_exact(ctx, m, k, n, bias):
    from franken_ocr_amd.engine import QInt8, linear_i8_dynamic

    _say(f"linear m={m} k={k} n={n} bias={bias}")
    seed = 9000 + m + k + n
    x = (synth.f32_normal(synth.seed_of(seed), m * k) * 3).reshape(m, k)
    x[0, :7] = 0.0
    w = synth.int8_uniform(synth.seed_of(seed + 1), n * k)
    ws = synth.f32_uniform(synth.seed_of(seed + 2), n, 1e-3, 2e-2)
    b = synth.f32_normal(synth.seed_of(seed + 3), n) if bias else None
    q = QInt8(w, ws, n, k, ctx)
    dy = ctx.empty((m, n), np.float32)
    linear_i8_dynamic(q, ctx.to_device(x), dy, None if b is None else ctx.to_device(b))
    st, want, _, _ = O.linear_i8_dynamic(x, w, ws, n, bias=b)
    assert st == 0
    got = dy.numpy()
    assert np.array_equal(got, want), f"{int((got != want).sum())} of {got.size} differ"


def test_linear_i8_dynamic_ties_even_known_answer(ctx):
    """nn.rs:601-628, zero-padded to k = 64 (zeros change neither the
    activation scale nor any sum): [0, 2, 0, 0], byte-identical on repeat."""
    from franken_ocr_amd.engine import QInt8, linear_i8_dynamic

    x = np.zeros((2, 64), np.float32)
    x[0, :8] = [-127.0, -2.5, -1.5, -0.5, 0.5, 1.5, 2.5, 127.0]
    w = np.zeros((2, 64), np.int8)
    w[0, 4] = 1
    w[1, 6] = 1
    q = QInt8(w.reshape(-1), np.ones(2, np.float32), 2, 64, ctx)
    dx = ctx.to_device(x)
    y1, y2 = ctx.empty((2, 2), np.float32), ctx.empty((2, 2), np.float32)
    linear_i8_dynamic(q, dx, y1)
    linear_i8_dynamic(q, dx, y2)
    assert y1.numpy().ravel().tolist() == [0.0, 2.0, 0.0, 0.0]
    assert np.array_equal(y1.numpy(), y2.numpy())


def test_quantize_rows_dynamic_rule_bit_exact(ctx):
    from franken_ocr_amd.engine import QUANT_DYNAMIC, quantize_rows_i8

    m, k = 37, 1280
    x = (synth.f32_normal(synth.seed_of(9100), m * k) * 5).reshape(m, k)
    x[3] = 0.0
    s = np.float32(np.abs(x[5]).max()) / np.float32(127.0)
    x[5, :64] = ((np.arange(64) - 32 + 0.5).astype(np.float32) * s).astype(np.float32)  # planted ties
    xq, xs = ctx.empty((m, k), np.int8), ctx.empty((m,), np.float32)
    quantize_rows_i8(ctx.to_device(x), xq, xs, rule=QUANT_DYNAMIC)
    for r in range(m):
        q, sc = O.quantize_row_dynamic(x[r])
        assert np.array_equal(xq.numpy()[r], q) and xs.numpy()[r] == sc, f"row {r}"


def test_linear_i8_dynamic_rejects_k_not_multiple_of_64(ctx):
    from franken_ocr_amd._abi import ContractViolation
    from franken_ocr_amd.engine import QInt8, linear_i8_dynamic

    q = QInt8(np.zeros(4 * 80, np.int8), np.ones(4, np.float32), 4, 80, ctx)
    with pytest.raises(ContractViolation, match="multiple of 64"):
        linear_i8_dynamic(q, ctx.to_device(np.zeros((2, 80), np.float32)), ctx.empty((2, 4), np.float32))


@pytest.fixture(scope="module")
def layer_w():
    from test_gpu_moe import make_layer

    return make_layer(9200)


@pytest.fixture(scope="module")
def gpu_layer(ctx, layer_w):
    from franken_ocr_amd.engine import MoeLayer

    return MoeLayer(H, I, E, K, *layer_w, ctx=ctx)


@pytest.mark.parametrize("t", [1, 24, 130])
def test_moe_prefill_i8_matches_oracle(ctx, gpu_layer, layer_w, t):
    _say(f"moe prefill i8 t={t}")
    x = synth.f32_normal(synth.seed_of(9300 + t), t * H).reshape(t, H)
    idx, gates = synth.zipf_routing(synth.seed_of(9400 + t), t, E, K)
    dout = ctx.empty((t, H), np.float32)
    dx, di, dg = ctx.to_device(x), ctx.to_device(idx), ctx.to_device(gates)
    gpu_layer.prefill(dx, di, dg, dout)
    st, want = O.moe_prefill_i8(x, idx, gates, *layer_w[1:], E, I)
    assert st == 0
    assert_rel(dout.numpy(), want, 1e-3)
    again = ctx.empty((t, H), np.float32)
    gpu_layer.prefill(dx, di, dg, again)
    assert np.array_equal(dout.numpy(), again.numpy())


@pytest.mark.parametrize("t", [130, 300])
def test_moe_prefill_i8_hot_expert_and_shared(ctx, layer_w, t):
    """Every token routed to the same six experts (t rows each: 64-row tiles
    per expert, the last one ragged) plus the shared expert, whose gate/up
    runs as extra units of the routed launch (3 and 5 row tiles)."""
    from franken_ocr_amd.engine import MoeLayer

    si = 1792
    _say(f"moe prefill i8 shared t={t}")
    x = synth.f32_normal(synth.seed_of(9500), t * H).reshape(t, H)
    idx = np.tile(np.array([[40, 3, 17, 63, 0, 9]], np.uint32), (t, 1))
    gates = synth.f32_uniform(synth.seed_of(9501), t * K, 0.05, 1.0).reshape(t, K)
    sw = [synth.int8_uniform(synth.seed_of(9502), si * H), synth.f32_uniform(synth.seed_of(9503), si, 1e-3, 2e-2),
          synth.int8_uniform(synth.seed_of(9504), si * H), synth.f32_uniform(synth.seed_of(9505), si, 1e-3, 2e-2),
          synth.int8_uniform(synth.seed_of(9506), H * si), synth.f32_uniform(synth.seed_of(9507), H, 1e-3, 2e-2)]
    L = MoeLayer(H, I, E, K, *layer_w, ctx=ctx)
    L.set_shared(si, *sw)
    dout = ctx.empty((t, H), np.float32)
    L.prefill(ctx.to_device(x), ctx.to_device(idx), ctx.to_device(gates), dout, with_shared=True)
    st, want = O.moe_prefill_i8(x, idx, gates, *layer_w[1:], E, I, shared=(si, *sw))
    assert st == 0
    assert_rel(dout.numpy(), want, 1e-3)


def test_moe_prefill_i8_plan_forms_agree(ctx, gpu_layer):
    """1400 tokens (8400 pairs) take the plan's round-by-round scatter, 700
    its barrier-free form for up to 8192 pairs; a token's output does not
    depend on the other tokens of the call (exact i32 sums per row, its own
    epilogue, its own ascending-expert combine), so one call over 1400 rows
    equals two calls over 700 bit for bit."""
    t = 1400
    _say(f"moe prefill i8 plan forms t={t}")
    x = synth.f32_normal(synth.seed_of(9600), t * H).reshape(t, H)
    idx, gates = synth.zipf_routing(synth.seed_of(9601), t, E, K)
    whole = ctx.empty((t, H), np.float32)
    gpu_layer.prefill(ctx.to_device(x), ctx.to_device(idx), ctx.to_device(gates), whole)
    halves = []
    for a, b in ((0, t // 2), (t // 2, t)):
        out = ctx.empty((b - a, H), np.float32)
        gpu_layer.prefill(ctx.to_device(x[a:b]), ctx.to_device(idx[a:b]), ctx.to_device(gates[a:b]), out)
        halves.append(out.numpy())
    assert np.array_equal(whole.numpy(), np.concatenate(halves))


def test_moe_prefill_i8_bad_expert_index(ctx, gpu_layer):
    from franken_ocr_amd._abi import ContractViolation

    t = 4
    idx = np.zeros((t, K), np.uint32)
    idx[2, 3] = E
    dout = ctx.empty((t, H), np.float32)
    with pytest.raises(ContractViolation, match="expert index out of range"):
        gpu_layer.prefill(ctx.to_device(np.ones((t, H), np.float32)), ctx.to_device(idx),
                          ctx.to_device(np.ones((t, K), np.float32)), dout)


@pytest.mark.parametrize("hidden,inter,si,t", [(192, 64, 320, 70), (320, 192, 64, 129), (1280, 896, 1792, 65)])
def test_moe_prefill_i8_narrow_down_blocks(ctx, hidden, inter, si, t):
    """Few rows take the down launch's 128-column blocks, the shared expert's
    among them: hidden sizes that fill them partly (192, 320 = 2.5 blocks) and
    K below, at and past a staged chunk, against the oracle (rel 1e-3, the MoE
    output's tolerance)."""
    from franken_ocr_amd.engine import MoeLayer

    n_e, k = 5, 2
    _say(f"moe prefill i8 narrow down H={hidden} I={inter} shared={si} t={t}")

    def mat(seed, *shape):
        return synth.int8_uniform(synth.seed_of(seed), int(np.prod(shape))).reshape(shape)

    def sc(seed, *shape):
        return synth.f32_uniform(synth.seed_of(seed), int(np.prod(shape)), 1e-3, 2e-2).reshape(shape)

    router = synth.f32_normal(synth.seed_of(9700), n_e * hidden, 0.0, 0.02).reshape(n_e, hidden)
    w = [mat(9701, n_e, inter, hidden), sc(9702, n_e, inter), mat(9703, n_e, inter, hidden), sc(9704, n_e, inter),
         mat(9705, n_e, hidden, inter), sc(9706, n_e, hidden)]
    sw = [mat(9707, si, hidden), sc(9708, si), mat(9709, si, hidden), sc(9710, si), mat(9711, hidden, si),
          sc(9712, hidden)]
    x = synth.f32_normal(synth.seed_of(9713), t * hidden).reshape(t, hidden)
    idx, gates = synth.zipf_routing(synth.seed_of(9714), t, n_e, k)
    layer = MoeLayer(hidden, inter, n_e, k, router, *w, ctx=ctx)
    layer.set_shared(si, *sw)
    out = ctx.empty((t, hidden), np.float32)
    layer.prefill(ctx.to_device(x), ctx.to_device(idx), ctx.to_device(gates), out, with_shared=True)
    flat = [a.reshape(-1) for a in w]
    st, want = O.moe_prefill_i8(x, idx, gates, *flat, n_e, inter, shared=(si, *[a.reshape(-1) for a in sw]))
    assert st == 0
    assert_rel(out.numpy(), want, 1e-3)


@pytest.mark.parametrize("m,k,n,bias", [
    (256, 64, 64, False),     # one K stage: three of a block's four waves add nothing
    (256, 1216, 65, True),    # a ring not filled, a column past the block
    (257, 1280, 127, False),  # the ring exactly full, one row in the last block
    (319, 1344, 1, True),     # one stage past the ring, one column
    (320, 2560, 192, False),  # two rings exactly
    (449, 2624, 640, True),   # and one stage more
    (448, 320, 4672, False),  # 7 x 73 blocks: 511
    (512, 320, 4096, False),  # 512
    (513, 320, 3648, False),  # 9 x 57: 513, past two blocks on each of 256 CUs
    (144, 1280, 1360, False),  # 765 of the GEMV's groups, three a CU
    (144, 1280, 1376, False),  # 774, one block row of 16 rows past the second
    (49, 1280, 3841, False),   # one row block of 49 rows
    (255, 1792, 1000, True),   # fewer than 256 rows with a bias
])
def test_linear_i8_small_blocks_bit_exact(ctx, m, k, n, bias):
    """64 x 64 blocks with K split over the waves: the i32 sums are exact in any
    order and the f32 formula is the oracle's, so no difference is allowed."""
    test_linear_i8_dynamic_bit_exact(ctx, m, k, n, bias)


def _hip():
    import ctypes

    path = next(ln.split()[-1] for ln in open("/proc/self/maps") if "libamdhip64" in ln)
    return ctypes.CDLL(path), ctypes


@pytest.mark.parametrize("m,k,n", [(256, 1280, 1280), (160, 1280, 1280), (159, 1280, 4096)])
def test_linear_i8_captured_before_the_tiled_weights(ctx, m, k, n):
    """A capture cannot allocate the tiled weight copy: a call recorded before
    the handle has one runs the kernel that needs none (the GEMV; the third
    shape is past its range and has had its 64-row-tile weights made by a call
    of few rows), and both give the oracle's bits."""
    from franken_ocr_amd.engine import QInt8, linear_i8_dynamic

    _say(f"captured linear m={m} k={k} n={n}")
    x = synth.f32_normal(synth.seed_of(9900 + m), m * k).reshape(m, k)
    w = synth.int8_uniform(synth.seed_of(9901), n * k)
    ws = synth.f32_uniform(synth.seed_of(9902), n, 1e-3, 2e-2)
    big = QInt8(w, ws, n, k, ctx)
    dx, dy = ctx.to_device(x), ctx.empty((m, n), np.float32)
    linear_i8_dynamic(big, dx, dy)  # the scratch, and the tiled route eagerly
    st, want, _, _ = O.linear_i8_dynamic(x, w, ws, n)
    assert st == 0 and np.array_equal(dy.numpy(), want)
    q = QInt8(w, ws, n, k, ctx)
    if n > 2048:
        zero = ctx.to_device(np.zeros(n, np.float32))
        linear_i8_dynamic(q, ctx.to_device(x[:5]), ctx.empty((5, n), np.float32), zero)
    dz = ctx.to_device(np.zeros((m, n), np.float32))
    _replays(ctx, lambda: linear_i8_dynamic(q, dx, dz), dz, want, 2)  # relaxed


def _replays(ctx, call, out, want, mode):
    """`call` captured in that mode, replayed three times."""
    hip, ct = _hip()
    stream, graph, ex = ct.c_void_p(ctx.stream()), ct.c_void_p(), ct.c_void_p()
    ctx.synchronize()
    assert hip.hipStreamBeginCapture(stream, mode) == 0
    try:
        call()
    finally:
        rc = hip.hipStreamEndCapture(stream, ct.byref(graph))
    assert rc == 0
    assert hip.hipGraphInstantiate(ct.byref(ex), graph, None, None, ct.c_size_t(0)) == 0
    for _ in range(3):
        out.copy_from(np.full(out.shape, 3.0, np.float32))
        assert hip.hipGraphLaunch(ex, stream) == 0
        ctx.synchronize()
        assert np.array_equal(out.numpy(), want)
    hip.hipGraphExecDestroy(ex)
    hip.hipGraphDestroy(graph)


@pytest.mark.parametrize("warm,m,k,n", [(64, 5, 1280, 4096), (255, 17, 1280, 1280), (256, 5, 128, 33000)])
def test_linear_i8_captured_with_the_tiled_weights_alone(ctx, warm, m, k, n):
    """A handle whose only call so far took the tiled order: a captured call of
    fewer rows, whose own order is the fragments', cannot make that copy and
    runs the tiled GEMM (the last shape in its 256-row blocks, five of them
    filled), with the oracle's bits."""
    from franken_ocr_amd.engine import QInt8, linear_i8_dynamic

    _say(f"captured linear m={m} after m={warm} k={k} n={n}")
    x = synth.f32_normal(synth.seed_of(9910 + m), warm * k).reshape(warm, k)
    w = synth.int8_uniform(synth.seed_of(9911), n * k)
    ws = synth.f32_uniform(synth.seed_of(9912), n, 1e-3, 2e-2)
    b = synth.f32_normal(synth.seed_of(9913), n)
    q, db, dx = QInt8(w, ws, n, k, ctx), ctx.to_device(b), ctx.to_device(x)
    warmed = ctx.empty((warm, n), np.float32)
    linear_i8_dynamic(q, dx, warmed, db)
    st, want, _, _ = O.linear_i8_dynamic(x, w, ws, n, b)
    assert st == 0 and np.array_equal(warmed.numpy(), want)
    dy = ctx.empty((m, n), np.float32)
    few = dx.view_rows(0, m)
    _replays(ctx, lambda: linear_i8_dynamic(q, few, dy, db), dy, want[:m], 0)  # global: no allocation at all
    linear_i8_dynamic(q, few, dy, db)  # and not captured
    assert np.array_equal(dy.numpy(), want[:m])


def test_linear_i8_first_calls_from_two_contexts(ctx):
    """Two threads, each with a context of its own, make a fresh handle's first
    calls at once: the tiled weight copy is made once and complete for both."""
    import threading

    from franken_ocr_amd import _abi
    from franken_ocr_amd.device import Context
    from franken_ocr_amd.engine import QInt8

    m, k, n = 64, 1280, 4096
    _say(f"first calls of two contexts m={m} k={k} n={n}")
    x = synth.f32_normal(synth.seed_of(9920), m * k).reshape(m, k)
    w = synth.int8_uniform(synth.seed_of(9921), n * k)
    ws = synth.f32_uniform(synth.seed_of(9922), n, 1e-3, 2e-2)
    st, want, _, _ = O.linear_i8_dynamic(x, w, ws, n)
    assert st == 0
    contexts = [Context(0), Context(0)]
    ins = [c.empty((m, k), np.float32).copy_from(x) for c in contexts]
    outs = [c.empty((m, n), np.float32) for c in contexts]
    for _ in range(4):
        q = QInt8(w, ws, n, k, ctx)
        ctx.synchronize()
        start, errors = threading.Barrier(2), []

        def call(i):
            try:
                start.wait()
                _abi.call("focr_hip_linear_i8_dynamic", contexts[i].handle, q.handle, ins[i].c_ptr, m, None,
                          outs[i].c_ptr)
                contexts[i].synchronize()
            except Exception as e:  # shown below, in the test's own thread
                errors.append(e)

        threads = [threading.Thread(target=call, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors, errors
        for out in outs:
            assert np.array_equal(out.numpy(), want)
        for c in contexts:
            c.synchronize()
        q.free()
    for a in (*ins, *outs):
        a.free()
    for c in contexts:
        c.close()
