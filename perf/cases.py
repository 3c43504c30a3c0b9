"""The work that users of this library have it do, as cases that can be timed.

Every case goes through the public entry points of the package.  Kinds:

  gemm      one block-scaled GEMM on operands that are already quantised (the launch of the reference's harness)
  linear    a projection layer as a model runs it: quantise this step's activations (1 x 128 groups), multiply
            with weights that were quantised when the model was loaded
  decode    a decode step: every projection of a layer on a small batch of tokens, recorded into a HIP graph once
            and replayed for every token, with a workspace of its own, as serving loops do
  weights   quantising a weight matrix (128 x 128 blocks) when a model is loaded or updated
  grouped   the experts of an MoE layer in one call: own rows and own weights per expert, common n and k
  host      the reference's host launcher: fp32 values in host memory in, bf16 in host memory out

Sizes: n and k of the projections are those of the reference's table of 18 shapes and of the five benchmark
configurations; the rows are a batch of tokens, from one to 8192, mostly no multiple of anything.
"""
import ctypes
import math
import random

import numpy as np
import torch

from __graft_entry__ import load_package

pkg = load_package()

# (n, k) of the projections in the reference's table (README.md:15-25)
PROJECTIONS = [(1536, 7168), (3072, 1536), (576, 7168), (7168, 256), (7168, 2048), (4608, 7168), (7168, 2304),
               (512, 7168), (4096, 512)]

# rows per expert: a ragged prefill of eight experts, and a decode step of 64 experts
PREFILL_EXPERTS = "509,1027,771,1533,250,2051,1023,1028"
DECODE_EXPERTS = ",".join(str(1 + (37 * i * i + 11 * i + 5) % 63) for i in range(64))

MOST_OPS = 8192 * 4608 * 7168     # m * n * k of the largest listed case
MOST_EXPERT_BYTES = 64 * 7168 * 2048


def listed():
    return [
        # one token through one projection: the smallest call, a loop of these runs at the rate of the launches
        {"name": "token", "kind": "gemm", "m": 1, "n": 7168, "k": 2048, "outliers": 0.0},
        # a decode batch of 32 through the same projection: weights streamed once for few operations
        {"name": "batch32", "kind": "gemm", "m": 32, "n": 7168, "k": 2048, "outliers": 0.0},
        # a decode step of 24 tokens: nine projections, each behind its quantiser, in one graph
        {"name": "decode_step", "kind": "decode", "m": 24},
        # a short prompt through a small projection: a few microseconds of work for a few CUs' worth of tiles
        {"name": "small_prefill", "kind": "gemm", "m": 1024, "n": 512, "k": 2048, "outliers": 0.0},
        # a prompt of a few hundred tokens, no round number of them, through a wide projection with its quantiser
        {"name": "ragged_prefill", "kind": "linear", "m": 333, "n": 4608, "k": 7168, "dtype": "bf16"},
        # a narrow projection with a long reduction: too few tiles for the chip unless K is split
        {"name": "narrow", "kind": "gemm", "m": 2048, "n": 576, "k": 7168, "outliers": 0.0},
        # a long prefill, quantiser and all: store-heavy, short reduction
        {"name": "long_prefill", "kind": "linear", "m": 8192, "n": 7168, "k": 2048, "dtype": "bf16"},
        # the largest: the headline configuration, activations with outliers
        {"name": "headline", "kind": "gemm", "m": 8192, "n": 4608, "k": 7168, "outliers": 0.01},
        # loading a model: one weight matrix
        {"name": "load_weights", "kind": "weights", "n": 4608, "k": 7168, "dtype": "bf16"},
        # an MoE layer in a prefill: eight experts with as many rows as the router gave each
        {"name": "moe_prefill", "kind": "grouped", "rows": PREFILL_EXPERTS, "n": 7168, "k": 2048},
        # an MoE layer in a decode step: 64 experts of 1 to 63 rows, all weights streamed once
        {"name": "moe_decode", "kind": "grouped", "rows": DECODE_EXPERTS, "n": 7168, "k": 2048},
        # the reference's host launcher on one shape of its table
        {"name": "host", "kind": "host", "m": 1024, "n": 1536, "k": 7168},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _projection(rng):
    """a projection of the table, or one of any other size (n and k in steps that weights come in)"""
    if rng.random() < 0.5:
        return rng.choice(PROJECTIONS)
    return 16 * _log_int(rng, 16, 512), 128 * _log_int(rng, 2, 64)


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "linear", "linear", "decode", "weights", "grouped", "grouped", "host"])
    n, k = _projection(rng)
    if kind == "decode":
        return {"kind": kind, "m": rng.randint(1, 64)}
    if kind == "weights":
        n = _log_int(rng, 256, 8192)
        return {"kind": kind, "n": n, "k": k, "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "grouped":
        groups = _log_int(rng, 2, 96)
        while groups * n * k > MOST_EXPERT_BYTES:
            groups -= 1
        groups = max(2, groups)
        if rng.random() < 0.5:
            lo, hi = 1, rng.choice([8, 16, 32, 64])
        else:
            lo, hi = 65, _log_int(rng, 128, 2048)
        rows = [rng.randint(lo, hi) for _ in range(groups)]
        while len(rows) > 2 and sum(rows) * n * k > MOST_OPS // 2:
            rows.pop()
        return {"kind": kind, "rows": ",".join(map(str, rows)), "n": n, "k": k}
    if kind == "host":
        while n > 256 and n * k > 4608 * 7168:
            n = n // 32 * 16
        return {"kind": kind, "m": _log_int(rng, 64, 2048), "n": n, "k": k}
    m = min(_log_int(rng, 1, 8192), MOST_OPS // (n * k))
    if rng.random() < 0.3:
        m = min(8192, -(-m // 64) * 64)     # batches that were padded to a round number
    if rng.random() < 0.05:
        n = max(1, n - rng.randint(1, 15))  # a table of any size
    if kind == "gemm":
        return {"kind": kind, "m": m, "n": n, "k": k, "outliers": rng.choice([0.0, 0.01])}
    return {"kind": kind, "m": m, "n": n, "k": k, "dtype": rng.choice(["bf16", "bf16", "f32"])}


# ---------------------------------------------------------------- inputs
DTYPES = {"bf16": (torch.bfloat16, pkg.DTYPE_BF16, 2), "f32": (torch.float32, pkg.DTYPE_F32, 4)}


def _values(gen, rows, k, dtype, outliers=0.0):
    x = torch.randn((rows, k), generator=gen, device="cuda", dtype=torch.float32)
    if outliers:
        x = torch.where(torch.rand((rows, k), generator=gen, device="cuda") < outliers, x * 50.0, x)
    return x.to(dtype)


def _quantised_a(gen, m, k, outliers=0.0):
    x = _values(gen, m, k, torch.bfloat16, outliers)
    a, s = _a_buffers(m, k)
    pkg.quantize_a_1x128(x, a, s, m, k, pkg.DTYPE_BF16, _stream())
    return a, s


def _quantised_b(gen, n, k):
    x = _values(gen, n, k, torch.bfloat16)
    b, s = _b_buffers(n, k)
    pkg.quantize_b_128x128(x, b, s, n, k, pkg.DTYPE_BF16, _stream())
    return b, s


def _a_buffers(m, k):
    return (torch.empty((k, m), dtype=torch.uint8, device="cuda"),
            torch.empty((k // 128, m), dtype=torch.float32, device="cuda"))


def _b_buffers(n, k):
    return (torch.empty((k, n), dtype=torch.uint8, device="cuda"),
            torch.empty((k // 128, (n + 127) // 128), dtype=torch.float32, device="cuda"))


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _rows(case):
    return [int(v) for v in case["rows"].split(",")]


# ---------------------------------------------------------------- one pass
def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return {"gemm": _prepare_gemm, "linear": _prepare_linear, "decode": _prepare_decode, "weights": _prepare_weights,
            "grouped": _prepare_grouped, "host": _prepare_host}[case["kind"]](case, gen, seed)


def run(state):
    return state["run"](state)


def _prepare_gemm(case, gen, seed):
    m, n, k = case["m"], case["n"], case["k"]
    a, sa = _quantised_a(gen, m, k, case["outliers"])
    b, sb = _quantised_b(gen, n, k)
    c = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    return {"run": _run_gemm, "args": (a, b, sa, sb, c, m, n, k), "stream": _stream()}


def _run_gemm(s):
    pkg.gemm(*s["args"], s["stream"])
    return s["args"][4]


def _prepare_linear(case, gen, seed):
    m, n, k = case["m"], case["n"], case["k"]
    dtype, code, _ = DTYPES[case["dtype"]]
    b, sb = _quantised_b(gen, n, k)
    x = _values(gen, m, k, dtype)
    a, sa = _a_buffers(m, k)
    c = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    return {"run": _run_linear, "quantise": (x, a, sa, m, k, code), "gemm": (a, b, sa, sb, c, m, n, k),
            "stream": _stream()}


def _run_linear(s):
    pkg.quantize_a_1x128(*s["quantise"], s["stream"])
    pkg.gemm(*s["gemm"], s["stream"])
    return {"a": s["gemm"][0], "a_scale": s["gemm"][2], "c": s["gemm"][4]}


def _prepare_decode(case, gen, seed):
    m = case["m"]
    opt = pkg.Options(flags=pkg.FLAG_WORKSPACE_ZEROED)
    need = max(pkg.workspace_bytes_ex(m, n, k, opt, any_alignment=True) for n, k in PROJECTIONS)
    ws = torch.zeros(max(need, 256), dtype=torch.uint8, device="cuda")
    layers = []
    for n, k in PROJECTIONS:
        b, sb = _quantised_b(gen, n, k)
        x = _values(gen, m, k, torch.bfloat16)
        a, sa = _a_buffers(m, k)
        layers.append((x, a, b, sa, sb, torch.empty((m, n), dtype=torch.bfloat16, device="cuda"), n, k))

    def step():
        st = _stream()
        for x, a, b, sa, sb, c, n, k in layers:
            pkg.quantize_a_1x128(x, a, sa, m, k, pkg.DTYPE_BF16, st)
            pkg.gemm_ex(a, b, sa, sb, c, m, n, k, opt, ws, ws.numel(), st)

    step()  # once outside the capture: the library looks its device over on the first call
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    return {"run": _run_decode, "graph": graph, "layers": layers, "workspace": ws}


def _run_decode(s):
    s["graph"].replay()
    return [layer[i] for layer in s["layers"] for i in (1, 3, 5)]


def _prepare_weights(case, gen, seed):
    n, k = case["n"], case["k"]
    dtype, code, _ = DTYPES[case["dtype"]]
    x = _values(gen, n, k, dtype)
    b, sb = _b_buffers(n, k)
    return {"run": _run_weights, "args": (x, b, sb, n, k, code), "stream": _stream()}


def _run_weights(s):
    pkg.quantize_b_128x128(*s["args"], s["stream"])
    return {"b": s["args"][1], "b_scale": s["args"][2]}


def _prepare_grouped(case, gen, seed):
    n, k, rows = case["n"], case["k"], _rows(case)
    a, b, sa, sb = [], [], [], []
    for m in rows:
        qa, s = _quantised_a(gen, m, k)
        a.append(qa)
        sa.append(s)
        qb, s = _quantised_b(gen, n, k)
        b.append(qb)
        sb.append(s)
    out = torch.empty((sum(rows), n), dtype=torch.bfloat16, device="cuda")  # the experts' rows one after the other
    c = list(out.split(rows))
    return {"run": _run_grouped, "args": (a, b, sa, sb, c, rows, n, k), "out": out, "stream": _stream()}


def _run_grouped(s):
    pkg.gemm_grouped(*s["args"], s["stream"])
    return s["out"]


def _prepare_host(case, gen, seed):
    m, n, k = case["m"], case["n"], case["k"]
    rng = np.random.default_rng(seed)
    values = lambda *shape: rng.random(shape, dtype=np.float32) * 10.0 - 5.0  # the harness's uniform values
    a, b = values(k, m), values(k, n)
    sa, sb = values(k // 128, m), values(k // 128, (n + 127) // 128)
    c = np.zeros((m, n), np.uint16)
    ptr = [ctypes.c_void_p(v.ctypes.data) for v in (c, a, b, sa, sb)]
    return {"run": _run_host, "arrays": (a, b, sa, sb), "c": c, "ptr": ptr, "size": (m, n, k)}


def _run_host(s):
    rc = pkg.lib().fp8_gemm_host(*s["ptr"], *s["size"], 0)
    if rc:
        raise pkg.Fp8GemmError(rc, "fp8_gemm_host")
    return torch.from_numpy(s["c"]).view(torch.bfloat16)


# ---------------------------------------------------------------- what a pass cannot do without
def _gemm_work(m, n, k):
    nkb = k // 128
    return (m * k + n * k + 4 * nkb * (m + (n + 127) // 128) + 2 * m * n, 2.0 * m * n * k)


def _quantise_work(rows, k, size, scales):
    return rows * k * (size + 1) + 4 * scales


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        byts, flops = _gemm_work(case["m"], case["n"], case["k"])
    elif kind == "linear":  # the quantised activations are an output of the first call and stay on the chip for the second
        m, n, k = case["m"], case["n"], case["k"]
        byts, flops = _gemm_work(m, n, k)
        byts += m * k * DTYPES[case["dtype"]][2]
    elif kind == "decode":
        byts = flops = 0.0
        for n, k in PROJECTIONS:
            b, f = _gemm_work(case["m"], n, k)
            byts += b + 2 * case["m"] * k
            flops += f
    elif kind == "weights":
        n, k = case["n"], case["k"]
        byts, flops = _quantise_work(n, k, DTYPES[case["dtype"]][2], (k // 128) * ((n + 127) // 128)), 0.0
    elif kind == "grouped":
        each = [_gemm_work(m, case["n"], case["k"]) for m in _rows(case)]
        byts, flops = sum(b for b, _ in each), sum(f for _, f in each)
    else:
        m, n, k = case["m"], case["n"], case["k"]
        byts, flops = _gemm_work(m, n, k)
        byts += 3 * (m * k + n * k)  # a and b come as fp32
    return {"bytes": float(byts), "flops": float(flops)}


def tolerance(case):
    """Quantised bytes and scales are fixed to the bit.  A GEMM's result is rounded to bf16 once: against the same
    sums in 64 bits (five shapes, one to 2048 rows) the 2-norm differs by 1.66e-3, the rounding itself, and no element
    by more than 4.0e-3 of the larger of itself and the root mean square; stated is four times that."""
    if case["kind"] == "weights":
        return "exact"
    return {"rel": 6.6e-3, "max": 1.6e-2, "differ": 0.0}
