"""GPU parity at the edges of the matmul dispatch: the shapes where one kernel takes over
from another, against the oracle's dequant and a float64 product."""
import sys

import numpy as np
import pytest

import arf_amd
from arf_amd import QType, arfq, synth

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def _want(oracle, qtype, x, raw, n):
    w = oracle.dequant(qtype, raw, n * x.shape[1]).reshape(n, x.shape[1])
    return x.astype(np.float64) @ w.T.astype(np.float64)


def _rel2(got, want):
    """|got - want| / |want| in the 2-norm."""
    return float(np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want))


@pytest.mark.parametrize("m,n,k", [(65, 4100, 512), (64 + 64, 512, 256), (129, 513, 2048), (333, 31, 1024)])
def test_iq4_xs_prefill_f32_x(gpu_ctx, oracle, m, n, k):
    # the direct-operand kernel: operands (ls - 32) * kv are exact to 2048 and rounded to
    # f16 above (half a unit in 12 bits, 2^-12 of the weight); x as hi + lo adds below 2^-21.
    # Independent errors of at most 2^-12 per product: the 2-norm stays under 2^-12.
    _say("case: iq4_xs prefill f32", m, n, k)
    raw, x = synth.weight("iq4_xs", n, k, seed=m + n), synth.activations(m, k, seed=m)
    x[:, ::37] *= 16
    w = gpu_ctx.upload(QType.IQ4_XS, raw, n, k)
    y = gpu_ctx.empty((m, n), np.float32)
    gpu_ctx.matmul(w, gpu_ctx.to_device(x), m, y)
    assert _rel2(y.numpy(), _want(oracle, "iq4_xs", x, raw, n)) <= 2.0 ** -12
    w.free()


def test_iq4_xs_noalloc_keeps_what_fits(gpu_ctx, oracle):
    # the direct kernel's partials for 32 tiles x 8 ranges exceed the fixed scratch: the
    # product still runs there, on the tile loop (weights rounded to f16: 2^-11 each)
    _say("case: iq4_xs noalloc")
    m, n, k = 100, 8192, 2048
    raw, x = synth.weight("iq4_xs", n, k, seed=3), synth.activations(m, k, seed=4)
    w, xd = gpu_ctx.upload(QType.IQ4_XS, raw, n, k), gpu_ctx.to_device(x)
    y = gpu_ctx.empty((m, n), np.float32)
    L = arf_amd.load_library()
    st = L.arfq_matmul_noalloc(gpu_ctx.handle, w.handle, 0, m, xd.ptr, int(arf_amd.DType.F32), y.ptr)
    assert st == arfq.ARFQ_OK, L.arfq_last_error(gpu_ctx.handle)
    assert _rel2(y.numpy(), _want(oracle, "iq4_xs", x, raw, n)) <= 2.0 ** -11
    w.free()


@pytest.mark.parametrize("x16", [False, True])
@pytest.mark.parametrize("qtype,m,n,k", [
    ("q6_k", 2, 70, 4096), ("q6_k", 4, 33, 3840), ("q6_k", 3, 40000, 256), ("q6_k", 3, 39000, 256),
    ("q8_0", 2, 1024, 16384), ("q8_0", 2, 1023, 16384), ("q8_0", 4, 7501, 1024), ("q8_0", 4, 7200, 1024),
    ("q8_0", 3, 4099, 4160)])
def test_small_m_q6_k_q8_0(gpu_ctx, oracle, qtype, m, n, k, x16):
    # both sides of the line between the f32 GEMVs and the skinny kernel (and k that only
    # the GEMV takes): exact products everywhere, f32 sums of at most 64 block sums of 8
    # sub-blocks, a random walk of 2^-24 steps below 2^-20.  ARFQ_OPT_GEMV_X16 has 16-bit
    # kernels for Q6_K at m = 2 only; the rest stays exact.  Its x is off by at most half a
    # step of 2^(e - 15), 2^e below twice the 32-element block's max, which is at most ~4
    # times its rms: 2^-16 * 8 / sqrt(3) of x, below 2^-13.
    _say("case: small m", qtype, m, n, k, x16)
    raw, x = synth.weight(qtype, n, k, seed=m + n), synth.activations(m, k, seed=m + k)
    if qtype == "q6_k":  # scales over all of i8
        rng = np.random.default_rng(n)
        raw.reshape(-1, 210)[:, 192:208] = rng.integers(0, 256, size=(raw.size // 210, 16), dtype=np.uint8)
    w = gpu_ctx.upload(QType[qtype.upper()], raw, n, k)
    y = gpu_ctx.empty((m, n), np.float32)
    gpu_ctx.set_options(arfq.OPT_GEMV_X16 if x16 else 0)
    try:
        gpu_ctx.matmul(w, gpu_ctx.to_device(x), m, y)
        got = y.numpy()
    finally:
        gpu_ctx.set_options(0)
    sixteen = x16 and qtype == "q6_k" and m == 2
    assert _rel2(got, _want(oracle, qtype, x, raw, n)) <= (2.0 ** -13 if sixteen else 2.0 ** -20)
    w.free()


@pytest.mark.parametrize("qtype,n,k", [
    ("q4_k", 1, 256), ("q4_k", 301, 9216), ("q5_k", 67, 768), ("q5_k", 5, 17408), ("q6_k", 70, 256),
    ("q6_k", 33, 4352), ("iq4_xs", 1030, 1792), ("iq4_xs", 64, 8448), ("q8_0", 50, 512), ("q8_0", 51000, 256),
    ("q8_0", 6211, 2304), ("q8_0", 19, 832), ("q8_0", 1001, 64), ("q4_k", 7, 38912), ("q6_k", 7, 40960)])
@pytest.mark.parametrize("x_dtype", [np.float32, np.float16])
def test_m1_x_types(gpu_ctx, oracle, qtype, n, k, x_dtype):
    # one x row, f32 or f16: exact products, f32 sums (lane and column sums, so chains of
    # far fewer than 2^8 terms: below 2^-20).  k of one block, of columns cut at every
    # length, past one x round, past the GEMVs' LDS; Q8_0 on both sides of its two
    # kernels' line and at k that is no multiple of 256.
    _say("case: m1", qtype, n, k, np.dtype(x_dtype).name)
    raw, x = synth.weight(qtype, n, k, seed=n + k), synth.activations(1, k, seed=n).astype(x_dtype)
    w = gpu_ctx.upload(QType[qtype.upper()], raw, n, k)
    y = gpu_ctx.empty((1, n), np.float32)
    gpu_ctx.matmul(w, gpu_ctx.to_device(x), 1, y)
    assert _rel2(y.numpy(), _want(oracle, qtype, x, raw, n)) <= 2.0 ** -20
    w.free()


def test_m1_q8_0_infinite_x(gpu_ctx, oracle):
    # an infinite x reaches its own row sums and no others: +-inf where its code is not 0,
    # NaN (0 * inf) where it is
    _say("case: q8_0 inf")
    n, k = 13000, 1280  # five blocks: the last column holds one
    raw, x = synth.weight("q8_0", n, k, seed=11), synth.activations(1, k, seed=12)
    x[0, k - 3] = np.inf
    w = gpu_ctx.upload(QType.Q8_0, raw, n, k)
    y = gpu_ctx.empty((1, n), np.float32)
    gpu_ctx.matmul(w, gpu_ctx.to_device(x), 1, y)
    wl = oracle.dequant("q8_0", raw, n * k).reshape(n, k)[:, k - 3]
    with np.errstate(invalid="ignore"):
        want = wl * np.float32(np.inf)
    assert np.array_equal(np.isnan(y.numpy()[0]), np.isnan(want))
    fine = ~np.isnan(want)
    assert np.array_equal(y.numpy()[0][fine], want[fine])
    w.free()


@pytest.mark.parametrize("qtype,n,k,x_dtype", [
    ("q6_k", 130, 256, np.float16), ("q6_k", 700, 4352, np.float16), ("iq4_xs", 1030, 1792, np.float16),
    ("iq4_xs", 3, 8448, np.float16), ("q8_0", 13000, 1280, np.float16), ("q8_0", 13000, 1280, np.float32)])
@pytest.mark.parametrize("at", [0, -3])
def test_m1_infinite_x(gpu_ctx, oracle, qtype, n, k, x_dtype, at):
    # +-inf by the sign of its weight, NaN (0 * inf) where that is 0, in one x row (f16; f32
    # for Q8_0, whose f32 GEMVs all multiply signed codes): the first block, or a last
    # column of one or three blocks
    _say("case: m1 inf", qtype, n, k, np.dtype(x_dtype).name, at)
    raw, x = synth.weight(qtype, n, k, seed=21), synth.activations(1, k, seed=22).astype(x_dtype)
    x[0, at] = -np.inf
    if x_dtype == np.float32:
        x[0, at ^ 1] = 3e38  # finite: beside the infinity it changes nothing
    w = gpu_ctx.upload(QType[qtype.upper()], raw, n, k)
    y = gpu_ctx.empty((1, n), np.float32)
    gpu_ctx.matmul(w, gpu_ctx.to_device(x), 1, y)
    with np.errstate(invalid="ignore"):
        want = oracle.dequant(qtype, raw, n * k).reshape(n, k)[:, at] * np.float32(-np.inf)
    assert np.array_equal(y.numpy()[0], want, equal_nan=True)
    w.free()


@pytest.mark.parametrize("qd", ["q6_k", "iq4_xs", "q8_0"])
def test_moe_pairs_infinite_h(gpu_ctx, oracle, qd):
    # one row of gate and up is not 0, and its g and u overflow h = silu(g) * u to inf: y is
    # +-inf by the sign of down's column of that row
    _say("case: moe inf", qd)
    E, hidden, inter, j = 2, 512, 1280, 1277
    gu = synth.weight("q8_0", inter, hidden, seed=31, experts=E).reshape(E, inter, hidden // 32, 34)
    gu[:, :, :, :2] = 0
    gu[:, j, :, 1] = 0x3C  # d = 1 in row j
    gu[:, j, :, 2:] = 1
    dn = synth.weight(qd, hidden, inter, seed=32, experts=E)
    ws = [gpu_ctx.upload(QType.Q8_0, gu.reshape(-1), inter, hidden, E) for _ in range(2)]
    ws.append(gpu_ctx.upload(QType[qd.upper()], dn, hidden, inter, E))
    ids, wts = np.array([[1]], np.int32), np.ones((1, 1), np.float32)
    x, y = np.full((1, hidden), 1e25, np.float32), gpu_ctx.empty((1, hidden), np.float32)
    gpu_ctx.moe_ids(*ws, gpu_ctx.to_device(ids), gpu_ctx.to_device(wts), 1, 1, gpu_ctx.to_device(x), y)
    with np.errstate(invalid="ignore"):
        want = oracle.dequant(qd, dn, E * hidden * inter).reshape(E, hidden, inter)[1, :, j] * np.float32(np.inf)
    assert np.array_equal(y.numpy()[0], want, equal_nan=True)
    for w in ws:
        w.free()


@pytest.mark.parametrize("qtype,m,n,k,wide", [("q8_0", 2, 4200, 3840, False), ("q8_0", 4, 1024, 16384, False),
                                              ("q6_k", 3, 130, 4352, True), ("q6_k", 4, 130, 4352, False),
                                              ("q6_k", 2, 17, 16384, True)])
def test_small_m_outlier_x(gpu_ctx, oracle, qtype, m, n, k, wide):
    # an x 2^30 above its row's others that meets weights of 0 leaves their products as
    # exact as f32 has them: the bound of test_small_m_q6_k_q8_0
    _say("case: small m outlier", qtype, m, n, k, wide)
    raw, x = synth.weight(qtype, n, k, seed=15), synth.activations(m, k, seed=16)
    at = k - 600
    if qtype == "q8_0":
        raw.reshape(n, k // 32, 34)[:, at // 32, 2 + at % 32] = 0  # the code
    else:
        b = raw.reshape(n, k // 256, 210)
        if wide:
            b[:, :, 192:208] = np.random.default_rng(n).integers(0, 256, size=(n, k // 256, 16), dtype=np.uint8)
        b[:, at // 256, 192 + at % 256 // 16] = 0  # the scale of its 16 elements
    x[0, at], x[1, at] = 2.0 ** 30, -(2.0 ** 30)
    w = gpu_ctx.upload(QType[qtype.upper()], raw, n, k)
    y = gpu_ctx.empty((m, n), np.float32)
    gpu_ctx.matmul(w, gpu_ctx.to_device(x), m, y)
    assert _rel2(y.numpy(), _want(oracle, qtype, x, raw, n)) <= 2.0 ** -20
    w.free()


@pytest.mark.parametrize("qtype,n,k,wide", [("q8_0", 4200, 3840, False), ("q6_k", 130, 4352, True),
                                            ("q6_k", 130, 4352, False)])
def test_small_m_infinite_x(gpu_ctx, oracle, qtype, n, k, wide):
    # an infinite x in the skinny kernel's three-part form: +-inf in its own row, NaN
    # (0 * inf) where its weight is 0, and the other rows as without it
    _say("case: small m inf", qtype, n, k, wide)
    m = 3
    raw, x = synth.weight(qtype, n, k, seed=13), synth.activations(m, k, seed=14)
    if wide:  # the form for scales over all of i8
        rng = np.random.default_rng(n)
        raw.reshape(-1, 210)[:, 192:208] = rng.integers(0, 256, size=(raw.size // 210, 16), dtype=np.uint8)
    x[1, k - 3] = np.inf
    w = gpu_ctx.upload(QType[qtype.upper()], raw, n, k)
    y = gpu_ctx.empty((m, n), np.float32)
    gpu_ctx.matmul(w, gpu_ctx.to_device(x), m, y)
    got, wl = y.numpy(), oracle.dequant(qtype, raw, n * k).reshape(n, k)[:, k - 3]
    with np.errstate(invalid="ignore"):
        want = wl * np.float32(np.inf)
    assert np.array_equal(np.isnan(got[1]), np.isnan(want))
    fine = ~np.isnan(want)
    assert np.array_equal(got[1][fine], want[fine])
    assert _rel2(got[[0, 2]], _want(oracle, qtype, x[[0, 2]], raw, n)) <= 2.0 ** -20
    w.free()


def _moe(gpu_ctx, oracle, qg, qd, tokens, top_k, hidden, inter, x_dtype):
    """moe_ids over four experts, the last id out of range, and the same in float64."""
    E = 4
    shapes = [(qg, inter, hidden), (qg, inter, hidden), (qd, hidden, inter)]
    raw = [synth.weight(q, n, k, seed=50 + i, experts=E) for i, (q, n, k) in enumerate(shapes)]
    ws = [gpu_ctx.upload(QType[q.upper()], r, n, k, E) for (q, n, k), r in zip(shapes, raw)]
    dq = [oracle.dequant(q, r, E * n * k).reshape(E, n, k).astype(np.float64) for (q, n, k), r in zip(shapes, raw)]
    rng = np.random.default_rng(tokens)
    x = (synth.activations(tokens, hidden, seed=7) * 0.05).astype(x_dtype)
    ids = rng.integers(0, E, size=(tokens, top_k)).astype(np.int32)
    wts = rng.random((tokens, top_k), dtype=np.float32)
    ids[-1, -1] = E
    y = gpu_ctx.empty((tokens, hidden), np.float32)
    gpu_ctx.moe_ids(*ws, gpu_ctx.to_device(ids), gpu_ctx.to_device(wts), tokens, top_k, gpu_ctx.to_device(x), y)
    want = np.zeros((tokens, hidden))
    for t in range(tokens):
        for e, wt in zip(ids[t], wts[t]):
            if e < E:
                g, u = dq[0][e] @ x[t].astype(np.float64), dq[1][e] @ x[t].astype(np.float64)
                with np.errstate(over="ignore"):
                    want[t] += wt * (dq[2][e] @ (g / (1 + np.exp(-g)) * u))
    for w in ws:
        w.free()
    return y.numpy(), want


@pytest.mark.parametrize("qg,qd,tokens,top_k,hidden,inter", [
    ("q4_k", "q6_k", 1, 2, 256, 512), ("q5_k", "q5_k", 3, 2, 768, 256), ("iq4_xs", "q6_k", 2, 3, 512, 1280),
    ("q8_0", "q8_0", 5, 1, 1280, 512), ("q6_k", "q4_k", 4, 2, 512, 768), ("iq4_xs", "iq4_xs", 1, 4, 4352, 256),
    ("q5_k", "q6_k", 70, 2, 512, 512), ("q8_0", "iq4_xs", 66, 2, 256, 256), ("q6_k", "q6_k", 70, 2, 256, 2048)])
@pytest.mark.parametrize("x_dtype", [np.float32, np.float16])
def test_moe_pairs_and_grouped(gpu_ctx, oracle, qg, qd, tokens, top_k, hidden, inter, x_dtype):
    # up to 128 pairs: the f32 GEMVs (each product's sums below 2^-20, g and u through
    # silu(g) * u and the down sums: four such errors, 2^-18).  More pairs: the grouped
    # kernels, x and h in f16 (2^-11 each).  One id of the given ones is out of range and
    # adds nothing.
    _say("case: moe", qg, qd, tokens, top_k, hidden, inter, np.dtype(x_dtype).name)
    got, want = _moe(gpu_ctx, oracle, qg, qd, tokens, top_k, hidden, inter, x_dtype)
    assert _rel2(got, want) <= (2.0 ** -18 if tokens * top_k <= 128 else 2.0 ** -10)


@pytest.mark.parametrize("q", ["q4_k", "q5_k", "q6_k", "iq4_xs", "q8_0"])
def test_moe_pairs_lds_past_64k(gpu_ctx, oracle, q):
    # x of gate and up, then of down, past the default LDS limit (16384 floats and their
    # sums) after a short one in the same process: each kernel raises its own limit.
    # The same bound as below 128 pairs above.
    for hidden, inter in [(512, 512), (16384, 256), (256, 16384)]:
        _say("case: moe lds", q, hidden, inter)
        got, want = _moe(gpu_ctx, oracle, q, q, 2, 1, hidden, inter, np.float32)
        assert _rel2(got, want) <= 2.0 ** -18


@pytest.mark.parametrize("qtype", ["q4_k", "q5_k", "q6_k", "iq4_xs", "q8_0"])
@pytest.mark.parametrize("n,k", [(4096, 1024), (3000, 5120)])
def test_f16_row_no_further_off_than_the_mfma_kernel(gpu_ctx, oracle, qtype, n, k):
    # the f32 GEMVs that take one f16 row are no further from 64 bits than the skinny MFMA
    # kernel, which takes the row beside a second one.  Over n outputs the two errors'
    # ratio is known to a few parts in sqrt(n)
    _say("case: f16 row error", qtype, n, k)
    raw = synth.weight(qtype, n, k, seed=41)
    x = np.repeat(synth.activations(1, k, seed=42).astype(np.float16), 2, axis=0)
    w = gpu_ctx.upload(QType[qtype.upper()], raw, n, k)
    y1, y2 = gpu_ctx.empty((1, n), np.float32), gpu_ctx.empty((2, n), np.float32)
    gpu_ctx.matmul(w, gpu_ctx.to_device(x[:1]), 1, y1)
    gpu_ctx.matmul(w, gpu_ctx.to_device(x), 2, y2)
    want = _want(oracle, qtype, x[:1], raw, n)
    assert _rel2(y1.numpy(), want) <= (1 + 4 / np.sqrt(n)) * _rel2(y2.numpy()[:1], want)
    w.free()


@pytest.mark.parametrize("m,n,k,wave", [(1, 1500, 30720, 1.16e-7), (3, 3000, 9216, 1.01e-7), (4, 1100, 30720, 1.19e-7)])
def test_q8_0_no_further_off_than_the_one_wave_gemv(gpu_ctx, oracle, m, n, k, wave):
    # the dot kernel at m = 1 and the skinny kernel at m = 2..4 add their columns and splits
    # so that a long row is no further from 64 bits than in gemv_q80w, which took these
    # products: `wave` is the lowest it measured over four such inputs (1.16 .. 1.23e-7,
    # 1.01 .. 1.05e-7, 1.19 .. 1.20e-7)
    _say("case: q8_0 long rows", m, n, k)
    raw, x = synth.weight("q8_0", n, k, seed=0), synth.activations(m, k, seed=50)
    w = gpu_ctx.upload(QType.Q8_0, raw, n, k)
    y = gpu_ctx.empty((m, n), np.float32)
    gpu_ctx.matmul(w, gpu_ctx.to_device(x), m, y)
    b = raw.reshape(n, k // 32, 34)  # the product of d and q in 64 bits, as the kernels have it
    wt = (b[:, :, :2].copy().view(np.float16).astype(np.float64) * b[:, :, 2:].view(np.int8)).reshape(n, k)
    assert _rel2(y.numpy(), x.astype(np.float64) @ wt.T) <= wave
    w.free()
