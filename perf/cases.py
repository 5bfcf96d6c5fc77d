"""The calls by which this library's speed is judged.

A case is one call, or one replayed chain of calls, of the public Python
surface (``hp_rms_norm_amd.ops``) on tensors that a transformer's serving or
prefill step has in hand.  ``listed()`` gives the named cases, ``draw()`` more
of the same ranges: 1 to 32768 rows (262144 for the per-head norm), 64 to
32768 elements a row, bfloat16 and float16, rows packed or padded, odd widths,
every output form of the fused op, the partial-sum form and the streamer.
"""
import math

import torch

import hp_rms_norm_amd as hp

EPS = 1e-6
FP8_MAX = 448.0
FLT_MIN = 1.17549435e-38
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
MX_FORMATS = {"mxfp8": hp.MXFP8, "mxfp4": hp.MXFP4}

# Ops and the entry point each stands for:
#   fused        hp_rms_norm (in place on input and residual)
#   graph        `calls` x hp_rms_norm captured in a HIP graph, replayed as one
#   fused_new    fused_add_rms_norm (new output and residual tensors)
#   fused_out    fused_add_rms_norm_out (the caller's tensors)
#   plain        rms_norm; with `heads`, on [tokens, heads, hidden]
#   fp8_row      fused_add_rms_norm_fp8 (new tensors, dynamic scale per row)
#   fp8_static   hp_rms_norm_fp8_static (one given scale)
#   fp8_group    fused_add_rms_norm_fp8_group (a scale per 128; `columns`:
#                token-minor scales)
#   mxfp8, mxfp4 hp_rms_norm_mx
#   reduce       reduce_add_rms_norm over `parts` partial sums
#   copy, relu   the streamer: hp.relu (a copy, as in the reference) and
#                hp.relu_max0


def listed():
    return [
        # one eager call of a small decode batch: launch and host cost.  1% of
        # the inputs are outliers, as activations have them
        dict(name="decode_eager", op="fused", rows=8, hidden=4096, dtype="bf16", outliers=True),
        # the norms of a decode step as serving engines run them, captured in
        # a graph: 16 of them over one residual stream, 32 tokens of 8192
        dict(name="decode_graph", op="graph", rows=32, hidden=8192, dtype="bf16", calls=16, outliers=True),
        # the headline shape: a prefill chunk of 4096 tokens, in place
        dict(name="prefill", op="fused", rows=4096, hidden=4096, dtype="bf16"),
        # the widest rows of the headline sweep, in place
        dict(name="prefill_wide", op="fused", rows=4096, hidden=32768, dtype="bf16"),
        # a ragged chunk, new output tensors: an eager module's forward
        dict(name="ragged_new", op="fused_new", rows=777, hidden=5120, dtype="bf16"),
        # an odd width in float16 (rows at every 2-byte offset)
        dict(name="odd_width", op="fused", rows=3000, hidden=4097, dtype="fp16"),
        # per-head norm of the queries: 4096 tokens x 32 heads of 128
        dict(name="per_head", op="plain", rows=131072, hidden=128, heads=32, dtype="bf16"),
        # the norm before a row-scaled FP8 GEMM
        dict(name="fp8_row", op="fp8_row", rows=2048, hidden=8192, dtype="bf16"),
        # the norm before a block-scaled FP8 GEMM, token-minor scales
        dict(name="fp8_group", op="fp8_group", rows=4096, hidden=7168, dtype="bf16", columns=True),
        # the norm before an MXFP4 GEMM, a large decode batch of wide rows
        dict(name="mxfp4", op="mxfp4", rows=512, hidden=16384, dtype="bf16"),
        # the second half of a one-shot 8-way tensor-parallel all-reduce
        dict(name="tp_reduce", op="reduce", rows=256, hidden=8192, dtype="bf16", parts=8),
        # the streaming companion on an MLP's activations
        dict(name="relu", op="relu", rows=4096, hidden=14336, dtype="fp16"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["fused"] * 5 + ["graph", "fused_new", "fused_out", "plain", "plain", "per_head", "fp8_row",
                                     "fp8_row", "fp8_static", "fp8_group", "fp8_group", "mxfp8", "mxfp4", "reduce",
                                     "reduce", "copy", "relu"])
    case = dict(op=op, dtype=rng.choice(["bf16", "bf16", "fp16"]))
    if op == "per_head":
        # heads of 64 to 256 elements
        case.update(op="plain", heads=rng.choice([1, 2, 4, 8, 16, 24, 32, 40, 64]), hidden=rng.choice([64, 96, 128, 192, 256]))
        case["rows"] = case["heads"] * _log_int(rng, 1, 4096)
        return case
    # widths: multiples of 128, as models have them, or (where the form takes
    # any width) anything
    unit = {"fp8_group": 128, "mxfp8": 32, "mxfp4": 32}.get(op, 1)
    if rng.random() < 0.75:
        hidden = 128 * _log_int(rng, 2, 256)
    else:
        hidden = unit * _log_int(rng, -(-64 // unit), 32768 // unit)
    # rows: as many as keep a pass at or under the widest listed case's work
    most = {"graph": 256}.get(op, 32768)
    parts = rng.choice([2, 4, 8]) if op == "reduce" else 1
    budget = 4096 * 32768 * 4 // (parts + 3) if op == "reduce" else 4096 * 32768
    case.update(rows=_log_int(rng, 1, max(1, min(most, budget // hidden))), hidden=hidden)
    if op == "reduce":
        case["parts"] = parts
    if op == "graph":
        case["calls"] = rng.choice([8, 16])
    if op == "fp8_group":
        case["columns"] = rng.random() < 0.5
    if op in ("fused", "fused_out", "plain", "copy", "relu") and rng.random() < 0.2:
        # rows of a wider buffer: input and output `pad` elements further apart
        case["pad"] = rng.choice([8, 64, 128, 1024])
    if case["dtype"] == "bf16" and rng.random() < 0.3:
        case["outliers"] = True
    return case


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + 17)


def _rows(case, g, outliers=False):
    """[rows, hidden] (with `pad`: a view of wider rows) of N(0, 1), with
    `outliers` 1% of the entries 50 times as large."""
    dtype = DTYPES[case["dtype"]]
    rows, hidden, pad = case["rows"], case["hidden"], case.get("pad", 0)
    t = torch.randn((rows, hidden + pad), generator=g, device="cuda", dtype=dtype)
    if outliers:
        t *= torch.where(torch.rand(t.shape, generator=g, device="cuda") < 0.01, 50.0, 1.0).to(dtype)
    return t[:, :hidden] if pad else t


def _inputs(case, seed):
    """The tensors a case's call reads, from the seed alone."""
    g, op, outliers = _generator(seed), case["op"], case.get("outliers", False)
    t = {}
    if op not in ("copy", "relu"):
        t["weight"] = (1.0 + 0.1 * torch.randn(case["hidden"], generator=g, device="cuda")).to(DTYPES[case["dtype"]])
    n = case.get("calls", case.get("parts", 1))
    t["inputs"] = [_rows(case, g, outliers) for _ in range(n)]
    if op not in ("plain", "copy", "relu"):
        t["residual"] = _rows(case, g)
    if op == "fp8_static":
        # calibrated on normalised rows: their largest magnitude is a few units
        t["scale"] = torch.full((1,), 6.0 / FP8_MAX, device="cuda")
    return t


def _capture(calls):
    """A graph of the calls; capturing runs none of them (the kernel is loaded
    by a call on other rows first)."""
    fn, (x, w, r, eps) = calls[0]
    fn(torch.zeros_like(x), w, torch.zeros_like(r), eps)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side):
            for fn, args in calls:
                fn(*args)
    torch.cuda.current_stream().wait_stream(side)
    return graph


def _buffer(case):
    """An output shaped and laid out like the case's rows."""
    t = torch.empty((case["rows"], case["hidden"] + case.get("pad", 0)), dtype=DTYPES[case["dtype"]], device="cuda")
    return t[:, :case["hidden"]] if case.get("pad") else t


def prepare(case, seed):
    """(function, arguments, outputs written by it or None if it returns them)."""
    t, op = _inputs(case, seed), case["op"]
    x = t["inputs"][0]
    w, r = t.get("weight"), t.get("residual")
    rows, hidden = case["rows"], case["hidden"]
    if op == "fused":
        return hp.hp_rms_norm, (x, w, r, EPS), (x, r)
    if op == "graph":
        graph = _capture([(hp.hp_rms_norm, (xi, w, r, EPS)) for xi in t["inputs"]])
        # (the graph reads w, x and r by address: the state keeps them)
        return graph.replay, (), (*t["inputs"], r, w)
    if op == "fused_new":
        return hp.fused_add_rms_norm, (x, r, w, EPS), None
    if op == "fused_out":
        out, res = _buffer(case), _buffer(case)
        return hp.fused_add_rms_norm_out, (out, res, x, w, r, EPS), (out, res)
    if op == "plain":
        out = _buffer(case)
        if case.get("heads"):
            x, out = (v.view(-1, case["heads"], hidden) for v in (x, out))
        return hp.rms_norm, (out, x, w, EPS), (out,)
    if op == "fp8_row":
        return _with_residual, (hp.fused_add_rms_norm_fp8, x, r, w, EPS), None
    if op == "fp8_static":
        q = torch.empty((rows, hidden), dtype=torch.float8_e4m3fn, device="cuda")
        return hp.hp_rms_norm_fp8_static, (q, t["scale"], x, w, r, EPS), (q, r)
    if op == "fp8_group":
        return _with_residual, (hp.fused_add_rms_norm_fp8_group, x, r, w, EPS, case["columns"]), None
    if op in MX_FORMATS:
        q = torch.empty((rows, hidden if op == "mxfp8" else hidden // 2), dtype=torch.uint8, device="cuda")
        scales = torch.empty((rows, hidden // 32), dtype=torch.uint8, device="cuda")
        return hp.hp_rms_norm_mx, (q, scales, x, w, r, EPS, MX_FORMATS[op]), (q, scales, r)
    if op == "reduce":
        out = _buffer(case)
        return hp.reduce_add_rms_norm, (out, t["inputs"], w, r, EPS), (out, r)
    out = _buffer(case)
    return (hp.relu if op == "copy" else hp.relu_max0), (out, x), (out,)


def _with_residual(fn, x, r, *rest):
    """The allocating quantised forms: their (q, scales) and the residual they update."""
    return (*fn(x, r, *rest), r)


def run(state):
    fn, args, outs = state
    got = fn(*args)
    return got if outs is None else outs


def work(case):
    """Every input element read once, every output element written once."""
    n, rows, hidden = case["rows"] * case["hidden"], case["rows"], case["hidden"]
    op = case["op"]
    if op in ("copy", "relu"):
        return {"bytes": 4 * n, "flops": n}
    calls = case.get("calls", 1)
    bytes_ = {"fused": 8 * n, "graph": 8 * n, "fused_new": 8 * n, "fused_out": 8 * n, "plain": 4 * n,
              "fp8_row": 7 * n + 4 * rows, "fp8_static": 7 * n + 4, "fp8_group": 7 * n + n // 32,
              "mxfp8": 7 * n + n // 32, "mxfp4": 6 * n + n // 2 + n // 32,
              "reduce": 2 * n * (case.get("parts", 1) + 3)}[op]
    # add, square and accumulate, two products; per part one more add
    return {"bytes": calls * (bytes_ + 2 * hidden), "flops": calls * n * (5 + case.get("parts", 1))}


def tolerance(case):
    if case["op"] in ("copy", "relu"):
        return "exact"
    # Another order of a row's binary32 sum moves a few in 10^5 of the 16-bit
    # outputs by one unit in the last place (measured over the ranges with the
    # widths' other lane mappings: rel 1.5e-5 in bfloat16, 5e-6 in float16);
    # in a small call one moved value weighs more.  The residual never moves.
    fp16 = case["dtype"] == "fp16"
    if case["op"].startswith("fp8"):
        # one 16-bit step can move an e4m3 code by one, 2^-3 of its value, and
        # that of a row's or group's maximum moves all of its codes' values
        return {"rel": 2e-3, "max": 0.15}
    if case["op"] in MX_FORMATS:
        # codes and block scales are bytes; the residual is exact
        return {"rel": 0.0, "max": 0.0, "differ": 1e-4}
    ulp = 2.0 ** (-10 if fp16 else -7)  # the largest step, relative
    return {"rel": max(3e-5 if fp16 else 1e-4, ulp / math.sqrt(case["rows"] * case["hidden"])), "max": 1.05 * ulp}


def _exact_norm(s, w):
    """s (already rounded to the tensors' type): its norm in 64 bits."""
    s = s.double()
    return s * torch.rsqrt(s.square().mean(-1, keepdim=True) + EPS) * w.double()


def exact(case, seed):
    t, op = _inputs(case, seed), case["op"]
    dtype = DTYPES[case["dtype"]]
    x = t["inputs"][0].double()
    if op == "copy":
        return (x,)
    if op == "relu":
        return (x.clamp(min=0),)
    w = t["weight"]
    if op == "plain":
        y = _exact_norm(x, w)
        return (y.view(-1, case["heads"], case["hidden"]) if case.get("heads") else y,)
    r = t["residual"].double()
    if op == "graph":
        outs = []
        for xi in t["inputs"]:
            s = xi.double() + r
            r = s.to(dtype).double()
            outs.append(_exact_norm(r, w))
        return (*outs, s, w.double())
    if op == "reduce":
        # the parts' sum is rounded once to the tensors' type
        x = torch.stack([p.double() for p in t["inputs"]]).sum(0).to(dtype).double()
    s = x + r
    y = _exact_norm(s.to(dtype), w)
    if op in ("fused", "fused_new", "fused_out", "reduce"):
        return (y, s)
    if op in MX_FORMATS:
        return (None, None, s)
    # FP8: the codes' values before rounding, of the 16-bit output
    y = y.to(dtype).double()
    if op == "fp8_static":
        return ((y / t["scale"].double()).clamp(-FP8_MAX, FP8_MAX), s)
    if op == "fp8_row":
        scale = (y.abs().amax(-1, keepdim=True) / FP8_MAX).clamp(min=FLT_MIN)
        return (y / scale, scale, s)
    groups = y.view(case["rows"], -1, 128)
    scales = (groups.abs().amax(-1, keepdim=True) / FP8_MAX).clamp(min=FLT_MIN)
    return ((groups / scales).view_as(y), scales.squeeze(-1), s)
