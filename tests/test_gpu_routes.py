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
