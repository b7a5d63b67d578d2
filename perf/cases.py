"""The work that programs have this library do, as measurable cases.

A case is one call of the library's host interface (arf_amd.Context): a quantized
matmul, the dense FFN block or the MoE block, over the range from the smallest decode
projection to a 2048-row prefill.  Weights are uploaded once, as a model's are; x and y
are device buffers (torch tensors here) that the call reads and writes.

Weight bytes are drawn on the GPU, block by block, with the distributions of
arf_amd/synth.py, except that Q6_K sub-block scales cover all of i8: quantizers put the
largest scale of every block at the end of the range.  Activations are normal with a few
channels sixteen times larger, as the residual stream of a language model has them.
"""
import math

import numpy as np
import torch

import arf_amd
from arf_amd import QType

# (weights per block, bytes per block)
BLOCK = {"q8_0": (32, 34), "q4_k": (256, 144), "q5_k": (256, 176), "q6_k": (256, 210), "iq4_xs": (256, 136)}
QTYPE = {"q8_0": QType.Q8_0, "q4_k": QType.Q4_K, "q5_k": QType.Q5_K, "q6_k": QType.Q6_K, "iq4_xs": QType.IQ4_XS}
# the IQ4 codebook (a table of the file format)
IQ4_VALUES = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)

ACTS = {"silu": None, "gelu": arf_amd.arfq.ACT_GELU_TANH}


def listed():
    return [
        # one projection of a small model, one token: launch and latency
        dict(name="q8_0 decode small", op="matmul", w="q8_0", m=1, n=2048, k=2048, x="f32"),
        # gate or up projection of a dense model, one token
        dict(name="q4_k decode", op="matmul", w="q4_k", m=1, n=17408, k=5120, x="f32"),
        # the vocabulary projection, one token: the largest matrix of a model
        dict(name="q6_k head decode", op="matmul", w="q6_k", m=1, n=151936, k=5120, x="f32"),
        # the FFN of one decode step, in the usual mix of formats (down in Q6_K)
        dict(name="ffn decode q4_k+q6_k", op="ffn", w="q4_k", down="q6_k", m=1, hidden=5120, inter=17408, act="silu"),
        # down projection for eight sequences, or eight drafted tokens
        dict(name="q6_k batch 8", op="matmul", w="q6_k", m=8, n=5120, k=17408, x="f32"),
        # gate projection for a ragged batch of sequences
        dict(name="q5_k batch 45", op="matmul", w="q5_k", m=45, n=17408, k=5120, x="f32"),
        # prompt of 2048 tokens, activations kept in f16
        dict(name="q4_k prefill 2048 f16", op="matmul", w="q4_k", m=2048, n=17408, k=5120, x="f16"),
        # a projection over a prompt of odd length, f32 activations
        dict(name="iq4_xs prefill 777", op="matmul", w="iq4_xs", m=777, n=4100, k=5120, x="f32"),
        # the FFN over a short prompt, f32 activations, the other gate activation
        dict(name="ffn prefill 333 gelu", op="ffn", w="q4_k", down="q6_k", m=333, hidden=4096, inter=11008, act="gelu"),
        # the MoE block for four sequences decoding
        dict(name="moe decode 4", op="moe", w="q4_k", down="q4_k", experts=128, topk=8, tokens=4, hidden=2048,
             inter=768, x="f32"),
        # the MoE block for a ragged batch, the usual mix of formats
        dict(name="moe batch 37 q4_k+q6_k", op="moe", w="q4_k", down="q6_k", experts=128, topk=8, tokens=37,
             hidden=2048, inter=768, x="f32"),
        # the MoE block over a prompt of 512 tokens
        dict(name="moe prefill 512", op="moe", w="q4_k", down="q4_k", experts=128, topk=8, tokens=512, hidden=2048,
             inter=768, x="f16"),
    ]


MAX_BYTES = 640e6  # weights of a drawn case: about the vocabulary projection's
MAX_FLOPS = 3.65e11  # the 2048-row prefill's; f32 activations take twice the matrix work


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: sizes spread over their logarithm, any row count, any format mix."""
    types = list(BLOCK)
    while True:
        op = rng.choice(["matmul", "matmul", "matmul", "ffn", "moe"])
        if op == "matmul":
            w = rng.choice(types)
            k = 64 * _log(rng, 8, 288) if w == "q8_0" else 256 * _log(rng, 2, 72)
            c = dict(op=op, w=w, m=_log(rng, 1, 2048), n=_log(rng, 512, 152064), k=k,
                     x=rng.choice(["f32", "f32", "f16"]))
        elif op == "ffn":
            w = rng.choice(types)
            c = dict(op=op, w=w, down=rng.choice([w, "q6_k"]), m=_log(rng, 1, 512), hidden=256 * _log(rng, 4, 24),
                     inter=256 * _log(rng, 8, 72), act=rng.choice(["silu", "gelu"]))
        else:
            w = rng.choice(["q4_k", "q4_k", "q8_0", "q5_k", "iq4_xs"])
            e = rng.choice([8, 16, 32, 64, 128])
            c = dict(op=op, w=w, down=rng.choice([w, w, "q6_k"]), experts=e, topk=rng.choice([2, 4, 8]),
                     tokens=_log(rng, 1, 512), hidden=256 * _log(rng, 4, 20), inter=256 * _log(rng, 2, 16),
                     x=rng.choice(["f32", "f16"]))
        f32 = c.get("x", "f32") == "f32"
        if sum(_tensor_bytes(t) for t in _tensors(c)) <= MAX_BYTES and work(c)["flops"] * (2 if f32 else 1) <= MAX_FLOPS:
            return c


def _tensors(c):
    """(format, rows, cols, experts) of the case's weights."""
    if c["op"] == "matmul":
        return [(c["w"], c["n"], c["k"], 1)]
    e = c.get("experts", 1)
    return [(c["w"], c["inter"], c["hidden"], e), (c["w"], c["inter"], c["hidden"], e),
            (c["down"], c["hidden"], c["inter"], e)]


def _tensor_bytes(t):
    fmt, n, k, e = t
    qk, nb = BLOCK[fmt]
    return e * n * k // qk * nb


def work(c):
    """Weights of every matrix (expert) that is used, x and y once each."""
    wb = sum(_tensor_bytes(t) for t in _tensors(c))
    if c["op"] == "matmul":
        rows, kin, nout, macs = c["m"], c["k"], c["n"], c["m"] * c["n"] * c["k"]
    elif c["op"] == "ffn":
        rows, kin, nout, macs = c["m"], c["hidden"], c["hidden"], 3 * c["m"] * c["hidden"] * c["inter"]
    else:
        e, t, kk = c["experts"], c["tokens"], c["topk"]
        wb *= 1 - (1 - kk / e) ** t  # the experts that some token picks
        rows, kin, nout, macs = t, c["hidden"], c["hidden"], 3 * t * kk * c["hidden"] * c["inter"]
    xb = 2 if c.get("x") == "f16" else 4
    return {"bytes": wb + rows * kin * xb + rows * nout * 4, "flops": 2.0 * macs}


def tolerance(c):
    """f32 sums: every path but these multiplies x (as f32, or as f16 parts that hold 22 bits
    and more) by the exact weights.  The MoE block's grouped GEMMs take x and h in f16 (3.8e-4
    measured against 64 bits), IQ4_XS prefill rounds its weights to f16 (2.1e-4); a decode
    step of Q4_K experts is f32 throughout."""
    if c["op"] == "moe":
        decode = c["tokens"] * c["topk"] <= 128 and c["w"] == c["down"] == "q4_k"
        return {"rel": 1e-5 if decode else 1.5e-3}
    if c["op"] == "matmul":
        return {"rel": 8e-4 if c["w"] == "iq4_xs" and c["m"] > 64 else 1e-5}
    return {"rel": 1.5e-3 if c["m"] > 64 and "iq4_xs" in (c["w"], c["down"]) else 1e-5}


# ---- a program's state ----------------------------------------------------------------


class Buffer:
    """A torch tensor as the binding takes device buffers: address, dtype and size."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()
        self.dtype = np.dtype({torch.float32: np.float32, torch.float16: np.float16}[t.dtype])


_context = None


def context():
    """One context for the process, as a program keeps one per device."""
    global _context
    if _context is None:
        torch.cuda.init()
        _context = arf_amd.Context(0)
    return _context


def _gen(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 64 + stream)
    return g


def _scale(g, n, s):
    v = torch.randn(n, generator=g, device="cuda").abs_().mul_(s).half()
    return v.view(torch.uint8).reshape(n, 2)


def _blocks(fmt, nblk, g):
    """Raw ggml blocks [nblk, bytes per block] (arf_amd/synth.py's distributions)."""
    b = torch.randint(0, 256, (nblk, BLOCK[fmt][1]), generator=g, device="cuda", dtype=torch.uint8)
    if fmt == "q8_0":
        b[:, 0:2] = _scale(g, nblk, 0.002)
        b[:, 2:] = torch.where(b[:, 2:] == 128, 127, b[:, 2:])  # codes in [-127, 127]
    elif fmt in ("q4_k", "q5_k"):
        b[:, 0:2] = _scale(g, nblk, 0.01)
        b[:, 2:4] = _scale(g, nblk, 0.01)
    elif fmt == "q6_k":
        b[:, 208:210] = _scale(g, nblk, 0.0012)
    else:
        b[:, 0:2] = _scale(g, nblk, 0.0005)
    return b


def _raw(c, seed):
    return [_blocks(t[0], _tensor_bytes(t) // BLOCK[t[0]][1], _gen(seed, 8 + i)) for i, t in enumerate(_tensors(c))]


def _x(c, seed):
    rows, k = (c["m"], c["k"]) if c["op"] == "matmul" else (c.get("m") or c["tokens"], c["hidden"])
    g = _gen(seed, 1)
    x = torch.randn(rows, k, generator=g, device="cuda")
    x *= torch.where(torch.rand(k, generator=g, device="cuda") < 1 / 128, 16.0, 1.0)
    return x.half() if c.get("x") == "f16" else x


def _logits(c, seed):
    return torch.randn(c["tokens"], c["experts"], generator=_gen(seed, 2), device="cuda")


def prepare(case, seed):
    ctx = context()
    x = _x(case, seed)
    s = {"case": case, "ctx": ctx, "x": Buffer(x)}
    s["w"] = [ctx.upload(QTYPE[fmt], raw.cpu().numpy(), n, k, e)
              for (fmt, n, k, e), raw in zip(_tensors(case), _raw(case, seed))]
    nout = case["n"] if case["op"] == "matmul" else case["hidden"]
    s["y"] = Buffer(torch.empty(x.shape[0], nout, device="cuda"))
    if case["op"] == "moe":
        s["logits"] = Buffer(_logits(case, seed))
    torch.cuda.synchronize()  # the context has a stream of its own
    return s


def run(s):
    c, ctx, x, y, w = s["case"], s["ctx"], s["x"], s["y"], s["w"]
    if c["op"] == "matmul":
        ctx.matmul(w[0], x, c["m"], y)
    elif c["op"] == "ffn":
        ctx.ffn(w[0], w[1], w[2], x, c["m"], y, ACTS[c["act"]])
    else:
        ctx.moe(w[0], w[1], w[2], s["logits"], c["tokens"], c["topk"], True, x, y)
    return y.t


# ---- the same in 64 bits --------------------------------------------------------------


def _f16(b):
    return b.contiguous().view(torch.float16).double()  # [nblk, 1]


def _six_bit(s):
    """Scales and mins of the eight sub-blocks from the 12 packed bytes: [nblk, 8] each."""
    a, b, c = s[:, 0:4], s[:, 4:8], s[:, 8:12]
    sc = torch.cat([a & 63, (c & 15) | (a >> 6) << 4], 1)
    mn = torch.cat([b & 63, (c >> 4) | (b >> 6) << 4], 1)
    return sc.double(), mn.double()


def _dequant(fmt, b):
    """Blocks [nblk, bytes] -> [nblk, weights per block] in 64 bits."""
    nb = b.shape[0]
    if fmt == "q8_0":
        return _f16(b[:, 0:2]) * b[:, 2:34].contiguous().view(torch.int8).double()
    if fmt in ("q4_k", "q5_k"):
        d, dmin = _f16(b[:, 0:2]), _f16(b[:, 2:4])
        sc, mn = _six_bit(b[:, 4:16])
        qs = b[:, -128:].reshape(nb, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(nb, 8, 32)  # 32 bytes hold two sub-blocks
        if fmt == "q5_k":
            bit = torch.arange(8, device=b.device, dtype=torch.uint8).reshape(1, 8, 1)
            q = q | ((b[:, 16:48].reshape(nb, 1, 32) >> bit) & 1) << 4
        return ((d * sc)[:, :, None] * q.double() - (dmin * mn)[:, :, None]).reshape(nb, 256)
    if fmt == "q6_k":
        ql, qh = b[:, 0:128].reshape(nb, 2, 2, 32), b[:, 128:192].reshape(nb, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)  # [nblk, half, quadrant, 32]
        two = torch.arange(0, 8, 2, device=b.device, dtype=torch.uint8).reshape(1, 1, 4, 1)
        q = (lo | ((qh >> two) & 3) << 4).reshape(nb, 16, 16).double() - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double() * _f16(b[:, 208:210])
        return (sc[:, :, None] * q).reshape(nb, 256)
    d = _f16(b[:, 0:2])
    hi = b[:, 2].int() | b[:, 3].int() << 8
    j = torch.arange(8, device=b.device)
    lo4 = (b[:, 4:8].int()[:, j // 2] >> (4 * (j % 2))) & 15
    ls = (lo4 | ((hi[:, None] >> (2 * j)) & 3) << 4).double() - 32
    qs = b[:, 8:136].reshape(nb, 8, 16)
    q = torch.cat([qs & 15, qs >> 4], 2)
    table = torch.tensor(IQ4_VALUES, device=b.device, dtype=torch.float64)
    return ((d * ls)[:, :, None] * table[q.long()]).reshape(nb, 256)


def _product(x, fmt, raw, n, k):
    """x [rows, k] . W[n, k]^T, in runs of weight rows."""
    per = k // BLOCK[fmt][0]
    step = max(1, (1 << 27) // k)
    return torch.cat([x @ _dequant(fmt, raw[r * per:min(r + step, n) * per]).reshape(-1, k).t()
                      for r in range(0, n, step)], 1)


def _glu(g, u, act):
    if act == "gelu":
        t = torch.clamp(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3), -15, 15)
        return 0.5 * g * (1 + torch.tanh(t)) * u
    return g * torch.sigmoid(g) * u


def exact(case, seed):
    x, raw, ts = _x(case, seed).double(), _raw(case, seed), _tensors(case)
    if case["op"] == "matmul":
        return _product(x, ts[0][0], raw[0], ts[0][1], ts[0][2])
    if case["op"] == "ffn":
        g, u = (_product(x, ts[i][0], raw[i], ts[i][1], ts[i][2]) for i in (0, 1))
        return _product(_glu(g, u, case["act"]), ts[2][0], raw[2], ts[2][1], ts[2][2])
    p = torch.softmax(_logits(case, seed).double(), 1)
    w, ids = torch.topk(p, case["topk"], 1)
    w = w / w.sum(1, keepdim=True)
    y = torch.zeros(case["tokens"], case["hidden"], device="cuda", dtype=torch.float64)
    for e in range(case["experts"]):
        t, slot = (ids == e).nonzero(as_tuple=True)
        if t.numel() == 0:
            continue
        one = [r.reshape(case["experts"], -1, r.shape[1])[e] for r in raw]
        g, u = (_product(x[t], ts[i][0], one[i], ts[i][1], ts[i][2]) for i in (0, 1))
        h = _glu(g, u, "silu")
        y.index_add_(0, t, w[t, slot, None] * _product(h, ts[2][0], one[2], ts[2][1], ts[2][2]))
    return y
