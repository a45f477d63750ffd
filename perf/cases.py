"""The calls whose speed counts: what programs built on this framework run.

A user's program keeps the coded matrices on the GPU and, for every token,
multiplies with them: single vectors
and small batches through RansMatrix.gemv and gemv_group, whole layers
through RansLinear, with prompts of some hundred rows through the same
module; it expands a matrix to bf16 with decode, or to its integer codes with
decode_codes; and data encoded in the reference's own layout runs on
ReferenceLayoutMatrix.  Encoding is not here: it runs on the host, once when
a model is converted, and its output's size depends on its input.

A case is a dict: "kind" (gemv, group, linear, decode, codes,
reflayout), rows and cols of the matrix (rows of each member for a group),
"bits" of entropy per code, "dist" of the weights, "esc", the share of codes
forced beyond the 8-bit range, "batch" rows of x, "dtype" of x, and for the
headline and the reference layout the tiling.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "vram-compression_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import rans  # noqa: E402
import rans_linear  # noqa: E402

MAX_WEIGHTS = 25600 * 5120


def _case(kind, rows, cols, bits=3.25, dist="laplace", esc=0.0, batch=1, dtype="bf16", **more):
    return dict(kind=kind, rows=rows, cols=cols, bits=bits, dist=dist, esc=esc, batch=batch,
                dtype=dtype, **more)


def listed():
    named = [
        # one token through the smallest projection of a 1.5B layer (o_proj):
        # the shortest call a token step makes, where its fixed cost counts
        ("o_proj 1536x1536 b1", _case("gemv", 1536, 1536)),
        # the repository's headline workload: down_proj of a 1.5B layer
        ("down 1536x8960 b1", _case("gemv", 1536, 8960, R=3, C=1792)),
        # q, k and v of a 1.5B layer: three matrices that share x, one call
        ("q/k/v 2048x1536 b1", _case("group", 1536, 1536, rows2=256, rows3=256)),
        # gate and up of a 1.5B layer with waterfilled steps and some
        # escapes, four sequences decoding at once
        ("gate/up 17920x1536 b4", _case("group", 8960, 1536, 2.25, esc=0.001, batch=4,
                                        rows2=8960, rows3=0)),
        # the largest matrices of the benchmark: 27B-class, heavy-tailed
        # codes with 1% escapes; one token, and four sequences on the
        # transposed shape
        ("27B gate 25600x5120 b1", _case("gemv", 25600, 5120, 2.25, "student3", 0.01)),
        ("27B down 5120x25600 b4", _case("gemv", 5120, 25600, 2.25, "student3", 0.01, batch=4)),
        # an uneven shard: a row count that few tile heights divide, columns
        # an odd multiple of 32, f32 activations, six sequences
        ("shard 1000x1568 b6 f32", _case("gemv", 1000, 1568, 4.25, "gauss", batch=6, dtype="f32")),
        # down_proj as nn.Linear, eight sequences decoding at once
        ("linear 1536x8960 8 rows", _case("linear", 1536, 8960, batch=8)),
        # an attention projection as nn.Linear, serving 32 sequences (or a
        # short prompt) at once
        ("linear 5120x5120 32 rows", _case("linear", 5120, 5120, 3.0, batch=32)),
        # a prompt of 512 tokens through an MLP projection
        ("linear 8960x1536 512 rows", _case("linear", 8960, 1536, 3.25, batch=512)),
        # a large matrix expanded to bf16, as prefill does and as a program
        # does that wants the dense weight
        ("decode 25600x5120", _case("decode", 25600, 5120, 2.25, "student3", 0.01)),
        # data encoded in the reference's layout, at its published tiling
        ("reference layout 1536x8960", _case("reflayout", 1536, 8960, 3.0, R=8, C=8960)),
    ]
    return [dict(c, name=n) for n, c in named]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _largest_prime(n):
    p, big = 2, 1
    while n > 1:
        while n % p == 0:
            n, big = n // p, p
        p += 1
    return big


def _shape(rng, most, row_unit=None):
    """rows x cols as layers and their shards have them: cols a multiple of
    32 without a large prime factor, rows mostly a multiple of 64, sometimes
    any number (those up to 4M weights)."""
    while True:
        cols = 32 * _log_uniform(rng, 8, 800)
        if _largest_prime(cols) > 37:
            continue
        unit = row_unit or (64 if rng.random() < 0.6 else 8 if rng.random() < 0.6 else 1)
        rows = unit * max(1, _log_uniform(rng, 256, 25600) // unit)
        if rows * cols <= (min(most, 4 << 20) if unit == 1 else most):
            return rows, cols


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "gemv", "group", "linear", "linear", "linear", "decode",
                       "codes", "reflayout"])
    dist = rng.choice(["laplace", "gauss", "student3"])
    bits = round(rng.uniform(2.0, 4.3), 2)
    esc = rng.choice([0.0, 0.0, 0.001, 0.01])
    dtype = rng.choice(["bf16", "bf16", "f32"])
    if kind == "gemv":
        rows, cols = _shape(rng, MAX_WEIGHTS)
        return _case(kind, rows, cols, bits, dist, esc, _log_uniform(rng, 1, 8), dtype)
    if kind == "group":
        cols = 64 * _log_uniform(rng, 8, 80)
        while _largest_prime(cols) > 37:
            cols = 64 * _log_uniform(rng, 8, 80)
        rows = [64 * _log_uniform(rng, 2, 140) for _ in range(2)]
        return _case(kind, rows[0], cols, bits, dist, esc, _log_uniform(rng, 1, 8), dtype,
                     rows2=rows[1], rows3=rng.choice([0, rows[1]]))
    if kind == "linear":
        rows, cols = _shape(rng, MAX_WEIGHTS // 4)
        return _case(kind, rows, cols, bits, dist, esc, _log_uniform(rng, 1, 1024), dtype)
    if kind == "reflayout":
        rows, cols = _shape(rng, 16 << 20, 64)
        R = rng.choice([1, 2, 4, 8, 16])
        C = 32 * rng.choice([d for d in range(1, cols // 32 + 1) if cols // 32 % d == 0])
        return _case(kind, rows, cols, bits, "laplace", 0.0, 1, dtype, R=R, C=C)
    rows, cols = _shape(rng, MAX_WEIGHTS // 2)
    return _case(kind, rows, cols, bits, dist, esc)


# --------------------------------------------------------------------- inputs
def _cdf(x, dist):
    if dist == "laplace":
        return np.where(x < 0, 0.5 * np.exp(np.minimum(x, 0)), 1 - 0.5 * np.exp(-np.maximum(x, 0)))
    if dist == "gauss":
        t = torch.from_numpy(np.asarray(x, np.float64)) / math.sqrt(2)
        return (0.5 * torch.erfc(-t)).numpy()
    u = x / math.sqrt(3)
    return 0.5 + (u / (1 + u * u) + np.arctan(u)) / math.pi


def _step_for(bits, dist):
    """The step whose quantised weights round(w/step) have `bits` bits of
    entropy."""
    k = np.arange(-4096, 4097) - 0.5
    lo, hi = -8.0, 3.0
    for _ in range(40):
        mid = (lo + hi) / 2
        p = np.diff(_cdf(k * math.exp(mid), dist))
        p = p[p > 0]
        h = float(-(p * np.log2(p)).sum())
        lo, hi = (mid, hi) if h > bits else (lo, mid)
    return math.exp((lo + hi) / 2)


def _codes(rows, cols, case, gen):
    """int32 codes on the GPU: quantised weights of the case's distribution,
    a share of them forced beyond the 8-bit range."""
    shape, kw = (rows, cols), dict(device="cuda", generator=gen)
    if case["dist"] == "laplace":
        w = torch.empty(shape, device="cuda").exponential_(generator=gen)
        w = torch.where(torch.rand(shape, **kw) < 0.5, -w, w)
    elif case["dist"] == "gauss":
        w = torch.randn(shape, **kw)
    else:
        q = torch.randn(shape, **kw).square_()
        q += torch.randn(shape, **kw).square_()
        q += torch.randn(shape, **kw).square_()
        w = torch.randn(shape, **kw).div_(q.div_(3).sqrt_())
        del q
    limit = 127 if case["kind"] == "reflayout" else 32767
    codes = w.div_(_step_for(case["bits"], case["dist"])).round_().clamp_(-limit, limit).int()
    del w
    if case["esc"]:
        big = torch.randint(128, 600, shape, dtype=torch.int32, **kw)
        big = torch.where(torch.rand(shape, **kw) < 0.5, -big, big)
        codes = torch.where(torch.rand(shape, **kw) < case["esc"], big, codes)
    return codes


def _draw_inputs(case, seed):
    """(codes of each matrix, steps of each, x, bias), all on the GPU: steps
    as waterfilling sets them per column, activations with some outlier
    channels."""
    gen = torch.Generator(device="cuda").manual_seed(1000003 * seed + 17)
    rows = [case["rows"]]
    if case["kind"] == "group":
        rows += [r for r in (case["rows2"], case["rows3"]) if r]
    cols = case["cols"]
    kw = dict(device="cuda", generator=gen)
    codes = [_codes(r, cols, case, gen) for r in rows]
    steps = [0.01 * torch.exp(0.5 * torch.randn(cols, **kw)) for _ in rows]
    x = torch.randn(case["batch"], cols, **kw)
    x *= torch.where(torch.rand(cols, **kw) < 0.005, 20.0, 1.0)
    if case["dtype"] == "bf16":
        x = x.bfloat16()
    if case["batch"] == 1:
        x = x[0]
    bias = 0.1 * torch.randn(rows[0], **kw)
    return codes, steps, x, bias


def prepare(case, seed):
    codes, steps, x, bias = _draw_inputs(case, seed)
    lib = rans.build()
    host = [c.cpu().numpy() for c in codes]
    del codes
    kind, cols = case["kind"], case["cols"]
    if kind == "reflayout":
        enc = rans.encode_reference_layout(host[0], case["R"], case["C"])
        m = rans.ReferenceLayoutMatrix(enc, steps[0].cpu(), lib)
        return dict(kind=kind, m=m, x=x)
    if kind == "linear":
        m = rans_linear.RansLinear.from_codes(host[0], steps[0].cpu(), bias, lib, tune=False)
        return dict(kind=kind, m=m, x=x)
    if kind == "group":
        tiling = rans.pick_group_tiling([len(h) for h in host], cols)
    elif "R" in case:
        tiling = case["R"], case["C"]
    else:
        tiling = rans.pick_tiling(case["rows"], cols)
    ms = [rans.RansMatrix(rans.encode(h, *tiling, 1), s.cpu(), lib) for h, s in zip(host, steps)]
    return dict(kind=kind, m=ms[0], ms=ms, x=x)


def run(state):
    kind = state["kind"]
    if kind in ("gemv", "reflayout"):
        return state["m"].gemv(state["x"])
    if kind == "group":
        return rans.gemv_group(state["ms"], state["x"])
    if kind == "linear":
        return state["m"](state["x"])
    if kind == "decode":
        return state["m"].decode()
    return state["m"].decode_codes()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "codes"):
        return None  # whole numbers, or bf16 values that have to be the same bit for bit
    codes, steps, x, bias = _draw_inputs(case, seed)
    ys = []
    for c, s in zip(codes, steps):
        xs = (x.double() * s.double()).reshape(-1, case["cols"])
        y = torch.empty(xs.shape[0], c.shape[0], dtype=torch.float64, device="cuda")
        for i in range(0, c.shape[0], 2048):
            y[:, i:i + 2048] = xs @ c[i:i + 2048].double().t()
        ys.append(y if x.dim() > 1 else y[0])
    if kind == "linear":
        return ys[0] + bias.double()
    return ys if kind == "group" else ys[0]


def work(case):
    """Coded weights and side table, steps and x read once, the result
    written once."""
    rows = case["rows"] + case.get("rows2", 0) + case.get("rows3", 0)
    cols, batch, kind = case["cols"], case["batch"], case["kind"]
    n = rows * cols
    coded = n * (case["bits"] / 8 + 4 * case["esc"])
    if kind in ("decode", "codes"):
        return {"bytes": coded + 4 * cols * (kind == "decode") + (2 if kind == "decode" else 4) * n,
                "flops": n}
    xsize = 2 if case["dtype"] == "bf16" else 4
    out = xsize if kind == "linear" else 4
    return {"bytes": coded + 4 * cols + batch * (cols * xsize + rows * out),
            "flops": 2 * n * batch}


def tolerance(case):
    kind = case["kind"]
    if kind in ("decode", "codes"):
        return "exact"
    if kind == "linear":
        # above some 16 rows the layer multiplies bf16 weights and returns
        # bf16 results: two roundings to 8 bits of every product and sum,
        # 3e-3 off the exact result where measured
        return {"rel": 1e-2, "max": 8e-2}
    # sums of f32 products: the order of summation is what differs
    return {"rel": 2e-6, "max": 4e-5}
