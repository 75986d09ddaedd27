"""The calls whose speed counts, through the package's public entry points.

A program that uses this backend compiles a fused group once (`hf.load`, or
`hf.DynamicGroup(..., runtime=True)` where the row count changes from call to
call), keeps it, and launches it on device tensors.  Each case is one such
group at one size.  Two kinds of use set the sizes: prompts and batches
(thousands of rows: bandwidth and matrix rate count) and token-by-token
decoding (a handful of rows: latency, launches and how well one small call
fills the chip count).

families
  vec_add      f32 elementwise add, 1-D
  rmsq         RMSNorm + dynamic per-token int8 quantisation, bf16 in
  softmax      safe softmax, f32 in, bf16 out
  argmax       reduce_with_index over a row of logits, f32
  w8a8         int8 contraction + per-token x per-channel dequant, bf16 out,
               weights [N, K] ("nk") or [K, N] ("kn")
  bf16         bf16 contraction, f32 sums, bf16 out
  mx           block-scaled fp8 / fp4 contraction, f32 out
  gemm_rmsq    an un-fused host function (int8 contraction -> scale -> RMSNorm
               -> int8 quant) split into a program of two groups
"rows": "runtime" takes the row count at launch (one code object for all).
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ascendnpu-ir_amd"))
import hfusion_mi355x as hf  # noqa: E402

# a row count no other dim of a drawn group has: with_dynamic_rows replaces it
_ANY_ROWS = 7919


def listed():
    return [
        # the elementwise integration group at its headline size: HBM streaming
        dict(name="vec_add_16m", fam="vec_add", n=1 << 24),
        # norm + quant of a prompt batch, the headline group
        dict(name="rmsq_prefill", fam="rmsq", rows=8192, cols=4096, rt="static"),
        # the same group while decoding a small batch: launch and row latency
        dict(name="rmsq_decode", fam="rmsq", rows=16, cols=4096, rt="runtime"),
        # softmax over long rows of scores
        dict(name="softmax_long", fam="softmax", rows=4096, cols=32768, rt="static"),
        # softmax over an odd row length (a sequence length is whatever it is)
        dict(name="softmax_odd", fam="softmax", rows=777, cols=5003, rt="static"),
        # greedy sampling of a decoding batch from a large vocabulary
        dict(name="argmax_decode", fam="argmax", rows=16, cols=152064, rt="static"),
        # a linear layer on a full prompt, quantised weights
        dict(name="w8a8_prefill", fam="w8a8", m=4096, n=4096, k=4096, layout="nk", rt="static"),
        # the same layer while decoding, token count known at launch only
        dict(name="w8a8_decode", fam="w8a8", m=16, n=4096, k=4096, layout="nk", rt="runtime"),
        # the layer on one ragged chunk of a prompt, weights as linalg.matmul has them
        dict(name="w8a8_chunk_kn", fam="w8a8", m=333, n=4096, k=4096, layout="kn", rt="static"),
        # a bf16 linear layer on a full prompt
        dict(name="bf16_prefill", fam="bf16", m=4096, n=4096, k=4096, layout="nk", rt="static"),
        # a block-scaled fp8 linear layer on a full prompt
        dict(name="mx_fp8_prefill", fam="mx", m=4096, n=4096, k=4096, fmt="e4m3"),
        # contraction, norm and quant handed over un-fused: a two-launch program
        dict(name="gemm_rmsq_program", fam="gemm_rmsq", m=512, n=4096, k=4096),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    fam = rng.choice(["vec_add", "rmsq", "softmax", "argmax", "w8a8", "w8a8", "w8a8", "bf16", "bf16", "mx", "mx", "gemm_rmsq"])
    if fam == "vec_add":
        return dict(fam=fam, n=_log_int(rng, 1 << 10, 1 << 24))
    if fam == "rmsq":
        return dict(fam=fam, rows=_log_int(rng, 1, 8192), cols=rng.choice([1024, 1536, 2048, 2560, 3072, 4096]),
                    rt=rng.choice(["static", "runtime"]))
    if fam == "softmax":
        return dict(fam=fam, rows=_log_int(rng, 1, 4096), cols=_log_int(rng, 64, 32768), rt="static")
    if fam == "argmax":
        return dict(fam=fam, rows=_log_int(rng, 1, 256), cols=_log_int(rng, 1000, 152064), rt="static")
    if fam == "gemm_rmsq":
        return dict(fam=fam, m=_log_int(rng, 1, 1024), n=rng.choice([1024, 2048, 4096]), k=128 * rng.randint(8, 32))
    # linear layers: token counts over the whole range, layer widths 1024 .. 4096
    m, n, k = _log_int(rng, 1, 4096), 16 * rng.randint(64, 256), 64 * rng.randint(16, 64)
    if fam == "mx":
        fmt = rng.choice(["e4m3", "e5m2", "e2m1"])
        return dict(fam=fam, m=m, n=n, k=256 * rng.randint(4, 16), fmt=fmt)
    layout, rt = rng.choice(["nk", "nk", "kn"]), rng.choice(["static", "runtime"])
    if layout == "kn" and rt == "runtime":
        k = (k + 127) // 128 * 128
    return dict(fam=fam, m=m, n=n, k=k, layout=layout, rt=rt)


def _group(case, build, rows):
    """The loaded group: compiled for these rows, or for any."""
    if case.get("rt") == "runtime":
        return hf.DynamicGroup(hf.groups.with_dynamic_rows(build(_ANY_ROWS), _ANY_ROWS), runtime=True)
    return hf.load(build(rows))


def _inputs(case, seed):
    """The device inputs of a case, made from the seed alone."""
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed * 1000003 + 17)

    def normal(shape, std=1.0):
        return torch.randn(shape, generator=gen, device=dev, dtype=torch.float32) * std

    def uniform(shape, lo, hi):
        return torch.rand(shape, generator=gen, device=dev, dtype=torch.float32) * (hi - lo) + lo

    def ints(shape, lo, hi, dtype):
        return torch.randint(lo, hi + 1, shape, generator=gen, device=dev, dtype=dtype)

    fam = case["fam"]
    if fam == "vec_add":
        return [uniform((case["n"],), -1.0, 1.0), uniform((case["n"],), -1.0, 1.0)]
    if fam == "rmsq":
        r, c = case["rows"], case["cols"]
        return [normal((r, c)).bfloat16(), uniform((c,), 0.5, 1.5).bfloat16()]
    if fam == "softmax":
        return [normal((case["rows"], case["cols"]), 2.0)]
    if fam == "argmax":
        x = normal((case["rows"], case["cols"]))
        # a duplicated row maximum now and then: the lowest index wins
        rows = torch.arange(0, case["rows"], 7, device=dev)
        x[rows, case["cols"] // 3] = x[rows].amax(dim=1)
        return [x]
    if fam == "gemm_rmsq":
        m, n, k = case["m"], case["n"], case["k"]
        return [ints((m, k), -127, 127, torch.int8), ints((n, k), -127, 127, torch.int8), uniform((n,), 0.5, 1.5).bfloat16()]
    m, n, k = case["m"], case["n"], case["k"]
    if fam == "mx":
        # e8m0 exponents around 2^0, as bytes
        sa, sb = (ints((r, k // 32), 120, 130, torch.uint8).view(torch.int8) for r in (m, n))
        if case["fmt"] == "e2m1":  # two values a byte along K
            return [ints((m, k // 2), -128, 127, torch.int8), ints((k // 2, n), -128, 127, torch.int8), sa, sb]
        dt = torch.float8_e4m3fn if case["fmt"] == "e4m3" else torch.float8_e5m2
        return [normal((m, k)).to(dt), normal((k, n)).to(dt), sa, sb]
    wshape = (n, k) if case["layout"] == "nk" else (k, n)
    if fam == "w8a8":
        return [ints((m, k), -127, 127, torch.int8), ints(wshape, -127, 127, torch.int8),
                uniform((m,), 0.001, 0.02), uniform((n,), 0.001, 0.02)]
    return [normal((m, k)).bfloat16(), normal(wshape, 1.0 / math.sqrt(k)).bfloat16()]  # bf16


def prepare(case, seed):
    g, fam, dev = hf.groups, case["fam"], torch.device("cuda:0")
    ins = _inputs(case, seed)

    def out(shape, dtype):
        return torch.empty(shape, dtype=dtype, device=dev)

    if fam == "vec_add":
        return hf.load(g.vec_add(case["n"])), ins + [out((case["n"],), torch.float32)]
    if fam == "rmsq":
        r, c = case["rows"], case["cols"]
        grp = _group(case, lambda rows: g.rmsnorm_quant(rows, c), r)
        return grp, ins + [out((r, c), torch.int8), out((r,), torch.float32)]
    if fam == "softmax":
        r, c = case["rows"], case["cols"]
        return _group(case, lambda rows: g.safe_softmax(rows, c), r), ins + [out((r, c), torch.bfloat16)]
    if fam == "argmax":
        r, c = case["rows"], case["cols"]
        return _group(case, lambda rows: g.argmax(rows, c), r), ins + [out((r,), torch.float32), out((r,), torch.int32)]
    m, n, k = case["m"], case["n"], case["k"]
    if fam == "gemm_rmsq":
        return hf.load(g.gemm_rmsnorm_quant(m, n, k)), ins + [out((m, n), torch.int8), out((m,), torch.float32)]
    if fam == "mx":
        f = case["fmt"]
        return hf.load(g.matmul_mx(m, n, k, fa=f, fb=f, via="format" if f == "e2m1" else "fp8")), ins
    build = g.w8a8_dequant if fam == "w8a8" else g.bf16_mmad
    grp = _group(case, lambda rows: build(rows, n, k, b_layout=case["layout"]), m)
    return grp, ins + [out((m, n), torch.bfloat16)]


def run(state):
    group, args = state
    return group(*args)


def work(case):
    fam = case["fam"]
    if fam == "vec_add":
        return {"bytes": 12 * case["n"], "flops": case["n"]}
    if fam in ("rmsq", "softmax", "argmax"):
        r, c = case["rows"], case["cols"]
        if fam == "rmsq":
            return {"bytes": 3 * r * c + 2 * c + 4 * r, "flops": 8 * r * c}
        if fam == "softmax":
            return {"bytes": 6 * r * c, "flops": 6 * r * c}
        return {"bytes": 4 * r * c + 8 * r, "flops": r * c}
    m, n, k = case["m"], case["n"], case["k"]
    flops = 2 * m * n * k
    if fam == "gemm_rmsq":
        return {"bytes": (m + n) * k + 2 * n + m * n + 4 * m, "flops": flops}
    if fam == "w8a8":
        return {"bytes": (m + n) * k + 4 * (m + n) + 2 * m * n, "flops": flops}
    if fam == "bf16":
        return {"bytes": 2 * (m + n) * k + 2 * m * n, "flops": flops}
    per = 0.5 if case["fmt"] == "e2m1" else 1
    return {"bytes": (m + n) * k * per + (m + n) * k // 32 + 4 * m * n, "flops": flops}


def tolerance(case):
    fam = case["fam"]
    if fam == "softmax":
        # f32 sums in another order move a few values by one bf16 rounding
        return {"rel": 1e-3, "max": 8e-3}
    if fam == "bf16":
        return {"rel": 1e-3, "max": 8e-3}  # as above: f32 sums, one rounding to bf16
    if fam == "mx":
        # fp8: the matrix core adds a 64-k block its own way (1.3e-5 from the
        # 64-bit product at 4096^3); fp4 products are exact and sum in f32
        return {"rel": 1e-5, "max": 1e-4} if case["fmt"] == "e2m1" else {"rel": 5e-5, "max": 5e-4}
    # integer sums, a fixed order of f32 sums, or one operation per element
    return "exact"


_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _mx_values(t, fmt, k_dim):
    """fp8 / fp4 operand as float64, K unpacked along k_dim."""
    if fmt != "e2m1":
        return t.float().double()
    table = torch.tensor(_E2M1 + [-v for v in _E2M1], dtype=torch.float64, device=t.device)
    b = t.view(torch.uint8).to(torch.int64)
    v = torch.stack([table[b & 15], table[b >> 4]], dim=k_dim + 1)
    shape = list(t.shape)
    shape[k_dim] *= 2
    return v.reshape(shape)


def exact(case, seed):
    fam = case["fam"]
    ins = _inputs(case, seed)
    d = [t.double() if t.dtype not in (torch.float8_e4m3fn, torch.float8_e5m2) else t for t in ins]
    if fam == "vec_add":
        return d[0] + d[1]
    if fam == "softmax":
        return torch.softmax(d[0], dim=1)
    if fam == "argmax":
        return (d[0].amax(dim=1), None)

    def scale_of(x, gamma):  # codes are whole numbers: their scale is what has a 64-bit value
        y = x * (x.square().mean(dim=1, keepdim=True) + 1e-6).rsqrt() * gamma
        return (None, y.abs().amax(dim=1) / 127.0)

    if fam == "rmsq":
        return scale_of(d[0], d[1])
    if fam == "gemm_rmsq":
        return scale_of((d[0] @ d[1].t().contiguous()) / 4096.0, d[2])
    if fam == "mx":
        a, b = _mx_values(ins[0], case["fmt"], 1), _mx_values(ins[1], case["fmt"], 0)
        sa, sb = (torch.exp2(t.view(torch.uint8).double() - 127.0).repeat_interleave(32, dim=1) for t in ins[2:])
        sb = sb.t()
        return (a * sa) @ (b * sb).contiguous()
    b = d[1].t().contiguous() if case["layout"] == "nk" else d[1]
    c = d[0] @ b
    return c * d[2][:, None] * d[3][None, :] if fam == "w8a8" else c
