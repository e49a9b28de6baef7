"""The calls whose speed matters: what a program on one MI355X asks of the C ABI, with the sizes it asks for.

listed() names the calls that stand for the work, draw() gives further ones of the same ranges, prepare() makes a call's
inputs on the GPU, run() makes the call, work() says what it cannot do without and tolerance() how far two correct
implementations may lie apart.  Run from the repository's root.
"""
import math
import os
import sys

import numpy as np
import torch

_PACKAGE = os.path.join(os.getcwd(), "pto-isa_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from pto_amd import capi, datagen  # noqa: E402

E4M3, E5M2, E2M1 = 0, 1, 4  # operand formats of the MX GEMMs (2 and 3 are the mixed forms of the first two)


def listed():
    return [
        # a small product, where launch and latency count: one layer of a small head
        {"name": "gemm_small", "path": "gemm", "m": 512, "n": 512, "k": 512},
        # an ordinary product whose rows and columns no tile divides
        {"name": "gemm_ragged", "path": "gemm", "m": 1000, "n": 3000, "k": 2048},
        # the benchmark's headline product
        {"name": "gemm_6144", "path": "gemm", "m": 6144, "n": 6144, "k": 6144},
        # the benchmark's MXFP8 product: e5m2 operands, bf16 result
        {"name": "mxfp8_6144", "path": "mx", "m": 6144, "n": 6144, "k": 6144, "format": E5M2, "c_fp32": False},
        # a linear layer in MXFP8: fp32 activations quantised on the way in, weights quantised beforehand
        {"name": "mxfp8_linear", "path": "mx_linear", "m": 1000, "n": 6144, "k": 4096},
        # the benchmark's MXFP4 product, ragged in m and n
        {"name": "mxfp4_ragged", "path": "mx", "m": 2040, "n": 8100, "k": 8192, "format": E2M1, "c_fp32": False},
        # attention over a whole sequence without a mask
        {"name": "fa_d128", "path": "fa", "batch": 1, "heads": 16, "seq_q": 4096, "seq_kv": 4096, "head_dim": 128, "causal": 0, "o_fp32": False},
        # causal prefill of a batch at head_dim 64
        {"name": "fa_causal_d64", "path": "fa", "batch": 4, "heads": 32, "seq_q": 2048, "seq_kv": 2048, "head_dim": 64, "causal": 1, "o_fp32": False},
        # prefill in chunks: 512 new tokens of one sequence that see themselves and the 1536 before them
        {"name": "fa_chunk", "path": "fa", "batch": 1, "heads": 16, "seq_q": 512, "seq_kv": 2048, "head_dim": 128, "causal": 1, "o_fp32": False},
        # the row-wise top-k of the reference's kernel: nearly a whole sort of every row
        {"name": "topk_1000", "path": "topk", "rows": 4800, "cols": 1024, "ld": 1280, "topk": 1000},
        # conversion of a tensor whose size no tile divides
        {"name": "cvt_bf16", "path": "cvt", "n": 2040 * 8100, "to": "bf16", "mode": capi.CAST_RINT},
        # embedding rows of a large batch of tokens
        {"name": "gather_f16", "path": "gather", "rows": 65536, "table_rows": 16384, "cols": 1024, "elem_bytes": 2},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _multiple(rng, lo, hi, of):
    return of * _log(rng, lo // of, hi // of)


def draw(rng):
    path = rng.choice(("gemm", "gemm", "mx", "mx_linear", "fa", "fa", "topk", "cvt", "gather"))
    if path == "gemm":
        if rng.random() < 0.25:  # few rows, or a contraction that is no multiple of 128: whole blocks in m and n
            return {"path": path, "m": _multiple(rng, 128, 2048, 128), "n": _multiple(rng, 256, 6144, 256), "k": _multiple(rng, 256, 6144, 32)}
        return {"path": path, "m": _log(rng, 192, 6144), "n": _multiple(rng, 128, 6144, 4), "k": _multiple(rng, 256, 6144, 128)}
    if path == "mx":
        fmt = rng.choice((E4M3, E5M2, 2, 3, E2M1, E2M1))
        return {"path": path, "m": _log(rng, 256, 6144), "n": _multiple(rng, 256, 6144, 4), "k": _multiple(rng, 512, 6144, 512),
                "format": fmt, "c_fp32": rng.random() < 0.5}
    if path == "mx_linear":
        return {"path": path, "m": _log(rng, 256, 4096), "n": _multiple(rng, 256, 6144, 4), "k": _multiple(rng, 512, 6144, 512)}
    if path == "fa":
        dim, causal = rng.choice((64, 128)), rng.choice((0, 1, 2))
        seq_q = _multiple(rng, 128, 4096, 128)
        seq_kv = seq_q if rng.random() < 0.5 else _multiple(rng, max(128, seq_q), 8192, 64)
        most = 16 * 4096 * 4096 * 128 // (seq_q * seq_kv * dim)  # (batch, head) pairs, by the work of the largest listed one
        heads = min(_log(rng, 4, 64), max(1, most))
        batch = min(_log(rng, 1, 8), max(1, most // heads))
        return {"path": path, "batch": batch, "heads": heads, "seq_q": seq_q, "seq_kv": seq_kv, "head_dim": dim, "causal": causal,
                "o_fp32": rng.random() < 0.25}
    if path == "topk":
        cols = _log(rng, 64, 4096)
        rows = min(_log(rng, 128, 8192), 4800 * 1024 // cols)
        return {"path": path, "rows": rows, "cols": cols, "ld": cols + rng.choice((0, 24, 256)), "topk": _log(rng, 1, cols)}
    if path == "cvt":
        to = rng.choice(("f16", "bf16"))
        mode = capi.CAST_RINT if to == "bf16" or rng.random() < 0.6 else rng.choice((capi.CAST_ROUND, capi.CAST_FLOOR, capi.CAST_CEIL, capi.CAST_TRUNC))
        return {"path": path, "n": _log(rng, 1 << 18, 1 << 27), "to": to, "mode": mode}
    elem = rng.choice((2, 4))
    cols = _multiple(rng, 32, 8192, 8)
    rows = min(_log(rng, 1024, 1 << 18), (1 << 27) // (cols * elem))
    return {"path": path, "rows": rows, "table_rows": min(_log(rng, 256, 1 << 17), (1 << 28) // (cols * elem)), "cols": cols, "elem_bytes": elem}


class _State:
    """What the program holds: the library, the stream it works on, inputs and outputs."""

    def __init__(self, case):
        self.lib = capi.load()
        self.stream = torch.cuda.current_stream().cuda_stream
        self.case = case


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _fp8(g, rows, cols, dtype):
    # the reference generator's distribution: uniform in [-5, 5), rounded
    return torch.empty((rows, cols), device="cuda").uniform_(-5.0, 5.0, generator=g).to(dtype).view(torch.uint8)


def _mx_operand(g, rows, k, fmt):
    if fmt == E2M1:  # integers in [-6, 6), two to a byte
        nibble = torch.from_numpy(datagen.fp8_encode(np.arange(-6, 6), E2M1)).cuda()
        v = nibble[torch.randint(0, 12, (rows, k // 2, 2), generator=g, device="cuda")]
        x = v[..., 0] | (v[..., 1] << 4)
    else:
        x = _fp8(g, rows, k, torch.float8_e4m3fn if fmt == E4M3 else torch.float8_e5m2)
    scale = torch.randint(127, 130, (rows, k // 32), generator=g, device="cuda", dtype=torch.uint8)
    return x.contiguous(), scale


def prepare(case, seed):
    s, g, path = _State(case), _generator(seed), case["path"]
    if path == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        s.a = torch.empty((m, k), device="cuda").uniform_(-1.0, 1.0, generator=g).half()
        s.b = torch.empty((n, k), device="cuda").uniform_(-1.0, 1.0, generator=g).half()
        s.c = torch.empty((m, n), dtype=torch.float32, device="cuda")
    elif path == "mx":
        fmt = case["format"]
        s.a, s.sa = _mx_operand(g, case["m"], case["k"], {2: E4M3, 3: E5M2}.get(fmt, fmt))
        s.b, s.sb = _mx_operand(g, case["n"], case["k"], {2: E5M2, 3: E4M3}.get(fmt, fmt))
        s.c = torch.empty((case["m"], case["n"]), dtype=torch.float32 if case["c_fp32"] else torch.bfloat16, device="cuda")
    elif path == "mx_linear":
        m, n, k = case["m"], case["n"], case["k"]
        s.x = torch.empty((m, k), device="cuda").normal_(generator=g)
        w = torch.empty((n, k), device="cuda").normal_(0.0, k ** -0.5, generator=g)
        s.q, s.sq = torch.empty((m, k), dtype=torch.uint8, device="cuda"), torch.empty((m, k // 32), dtype=torch.uint8, device="cuda")
        s.b, s.sb = torch.empty((n, k), dtype=torch.uint8, device="cuda"), torch.empty((n, k // 32), dtype=torch.uint8, device="cuda")
        s.c = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
        capi.check(s.lib.pto_quant_mxfp8_f32(s.stream, s.b.data_ptr(), s.sb.data_ptr(), w.data_ptr(), n, k), "pto_quant_mxfp8_f32")
    elif path == "fa":
        q = (case["batch"], case["heads"], case["seq_q"], case["head_dim"])
        kv = (case["batch"], case["heads"], case["seq_kv"], case["head_dim"])
        s.q, s.k, s.v = (torch.empty(shape, device="cuda").normal_(generator=g).half() for shape in (q, kv, kv))
        s.o = torch.empty(q, dtype=torch.float32 if case["o_fp32"] else torch.float16, device="cuda")
        s.lse = torch.empty(q[:3], dtype=torch.float32, device="cuda")
    elif path == "topk":
        rows, k = case["rows"], case["topk"]
        s.src = torch.empty((rows, case["ld"]), device="cuda").normal_(generator=g)
        s.ids = torch.arange(case["cols"], dtype=torch.int32, device="cuda")
        s.score, s.index = torch.empty((rows, k), device="cuda"), torch.empty((rows, k), dtype=torch.int32, device="cuda")
    elif path == "cvt":
        s.x = torch.empty(case["n"], device="cuda").normal_(0.0, 100.0, generator=g)
        odd = torch.tensor([math.inf, -math.inf, math.nan, 65519.996, 65520.0, 1e-40, -1e-7, 6.1e-5, 0.0, -0.0, 3e38], device="cuda")
        at = torch.randint(0, case["n"], (max(1, case["n"] // 1000),), generator=g, device="cuda")
        s.x[at] = odd[at % odd.numel()]
        s.y = torch.empty(case["n"], dtype=torch.int16, device="cuda")  # bit patterns
    else:
        dtype = torch.int16 if case["elem_bytes"] == 2 else torch.int32
        top = torch.iinfo(dtype).max
        s.table = torch.randint(-top, top, (case["table_rows"], case["cols"]), generator=g, dtype=dtype, device="cuda")
        s.ids = torch.randint(0, case["table_rows"], (case["rows"],), generator=g, dtype=torch.int32, device="cuda")
        s.out = torch.empty((case["rows"], case["cols"]), dtype=dtype, device="cuda")
    return s


def run(s):
    case, lib, path = s.case, s.lib, s.case["path"]
    if path == "gemm":
        capi.check(lib.pto_gemm_f16f32(s.stream, s.c.data_ptr(), s.a.data_ptr(), s.b.data_ptr(), case["m"], case["n"], case["k"]), "pto_gemm_f16f32")
        return s.c
    if path == "mx":
        args = (s.stream, s.c.data_ptr(), s.a.data_ptr(), s.b.data_ptr(), s.sa.data_ptr(), s.sb.data_ptr(), case["m"], case["n"], case["k"])
        if case["format"] == E2M1:
            capi.check(lib.pto_gemm_mxfp4(*args, int(case["c_fp32"])), "pto_gemm_mxfp4")
        else:
            capi.check(lib.pto_gemm_mxfp8(*args, case["format"], int(case["c_fp32"])), "pto_gemm_mxfp8")
        return s.c
    if path == "mx_linear":
        m, n, k = case["m"], case["n"], case["k"]
        capi.check(lib.pto_quant_mxfp8_f32(s.stream, s.q.data_ptr(), s.sq.data_ptr(), s.x.data_ptr(), m, k), "pto_quant_mxfp8_f32")
        capi.check(lib.pto_gemm_mxfp8(s.stream, s.c.data_ptr(), s.q.data_ptr(), s.b.data_ptr(), s.sq.data_ptr(), s.sb.data_ptr(), m, n, k, E4M3, 0),
                   "pto_gemm_mxfp8")
        return {"q": s.q, "scale": s.sq, "c": s.c}
    if path == "fa":
        capi.check(lib.pto_fa_fwd_f16(s.stream, s.o.data_ptr(), s.lse.data_ptr(), s.q.data_ptr(), s.k.data_ptr(), s.v.data_ptr(), case["batch"],
                                      case["heads"], case["seq_q"], case["seq_kv"], case["head_dim"], case["causal"], int(case["o_fp32"])),
                   "pto_fa_fwd_f16")
        return {"o": s.o, "lse": s.lse}
    if path == "topk":
        capi.check(lib.pto_topk_f32(s.stream, s.score.data_ptr(), s.index.data_ptr(), s.src.data_ptr(), s.ids.data_ptr(), case["rows"], case["cols"],
                                    case["ld"], case["topk"]), "pto_topk_f32")
        return {"score": s.score, "index": s.index}
    if path == "cvt":
        call = lib.pto_tcvt_f32_f16 if case["to"] == "f16" else lib.pto_tcvt_f32_bf16
        capi.check(call(s.stream, s.y.data_ptr(), s.x.data_ptr(), case["n"], case["mode"]), "pto_tcvt_f32_" + case["to"])
        return s.y
    capi.check(lib.pto_gather_rows(s.stream, s.out.data_ptr(), s.table.data_ptr(), s.ids.data_ptr(), case["rows"], case["table_rows"], case["cols"],
                                   case["elem_bytes"]), "pto_gather_rows")
    return s.out


def work(case):
    path = case["path"]
    if path == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * (m + n) * k + 4 * m * n, "flops": 2 * m * n * k}
    if path == "mx":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": (m + n) * (k // (2 if case["format"] == E2M1 else 1) + k // 32) + (4 if case["c_fp32"] else 2) * m * n, "flops": 2 * m * n * k}
    if path == "mx_linear":  # activations read once; their fp8 form, which the caller gets as well, written once
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * m * k + (m + n) * (k + k // 32) + 2 * m * n, "flops": 2 * m * n * k}
    if path == "fa":
        pairs, sq, skv, d = case["batch"] * case["heads"], case["seq_q"], case["seq_kv"], case["head_dim"]
        seen = sq * skv
        if case["causal"]:
            first = 1 + (skv - sq if case["causal"] == 1 else 0)  # keys that the first query sees
            seen = sum(min(skv, first + i) for i in range(sq))
        return {"bytes": pairs * (2 * d * (sq + 2 * skv) + (4 if case["o_fp32"] else 2) * d * sq + 4 * sq), "flops": 4 * pairs * seen * d}
    if path == "topk":
        return {"bytes": 4 * case["rows"] * case["cols"] + 4 * case["cols"] + 8 * case["rows"] * case["topk"], "flops": 0}
    if path == "cvt":
        return {"bytes": 6 * case["n"], "flops": 0}
    width = case["cols"] * case["elem_bytes"]  # a table smaller than the batch is read once, whole
    return {"bytes": case["rows"] * (width + 4) + min(case["rows"], case["table_rows"]) * width, "flops": 0}


def tolerance(case):
    # about four times what these paths differ by from the same call in 64 bits, rounded to the result's type
    path = case["path"]
    if path == "gemm":  # measured: rel 5e-7, max 4.5e-6 at k = 6144
        return {"rel": 2e-6, "max": 2e-5}
    if path == "mx" and case["c_fp32"]:  # measured: rel 1.1e-5, max 6e-5 (the matrix instruction adds with about 20 bits)
        return {"rel": 4e-5, "max": 2.4e-4}
    if path in ("mx", "mx_linear"):  # measured: rel 2.4e-4, max one step of bf16 (2^-7) where the sum is near a tie
        return {"rel": 1e-3, "max": 1.6e-2}
    if path == "fa":  # measured: rel 3e-4, max 1.6e-3 (fp16 probabilities)
        return {"rel": 1.2e-3, "max": 6.4e-3}
    return "exact"
