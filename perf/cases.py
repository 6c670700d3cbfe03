"""The work this library is timed on: calls of its operators as a tensor-parallel serving program makes them.

`listed()` names the cases, `draw()` gives more of the same ranges, `prepare()` makes what a program has in hand before
the call (operands, staged peers, output, workspace, plan), `run()` is one call of a public operator, `work()` the bytes
and operations the operator cannot do without, `tolerance()` what another correct implementation may differ by.

Sizes: P ranks (tensor parallel), m tokens, k = this rank's share of the reduction, n output columns.  Decode batches are
small and of any size, prefill chunks large; k and n are what a weight matrix leaves after sharding, mostly whole cache
lines, sometimes not.  Reduce-scatter calls store the other ranks' tiles to the symmetric workspace, which the peers pull,
except where the case folds them into checksums as the benchmark does.
"""
import ctypes
import math

import torch

from mm_rs_with_catlass_amd import lib, ops

DEV = "cuda:0"
_DT = {"fp16": torch.float16, "bf16": torch.bfloat16}
_COUNTERS = lib.WORKSPACE_COUNTER_BYTES


def _case(name, op, m, k, n, ranks, rank, dtype, trans_b, **more):
    """op: allreduce / allgather / reduce_scatter (float), quant_reduce_scatter / quant_decode / quant_pipelined (W8A8).
    dtype: the element type of the float operators, the output type of the W8A8 ones.  kept: rows this rank keeps
    (quant_decode).  outbound: the other ranks' tiles are stored, not summed.  bound: the call's arguments are bound once
    and the program repeats the launch."""
    c = {"op": op, "m": m, "k": k, "n": n, "ranks": ranks, "rank": rank, "dtype": dtype, "trans_b": trans_b,
         "bias": False, "kept": 0, "outbound": False, "int32_reduce": False, "bound": False}
    c.update(more)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # one token of one request through a W8A8 projection stored output-major; a serving loop repeats the bound launch
        _case("quant_decode_1", "quant_decode", 1, 8192, 8192, 8, 0, "bf16", True, kept=1, bound=True),
        # a full decode batch against row-major weights; this rank keeps its eighth
        _case("quant_decode_64", "quant_decode", 64, 8192, 8192, 8, 0, "bf16", False, kept=8),
        # a mixed batch (decode rows and the end of a prefill) that is no multiple of anything; every row is kept (all-reduce)
        _case("quant_decode_203", "quant_decode", 203, 1792, 4096, 8, 0, "bf16", True, kept=203, bias=True),
        # decode of an unquantised model: row-parallel projection, every rank needs every row
        _case("allreduce_decode_16", "allreduce", 16, 1024, 8192, 8, 3, "bf16", True),
        # a short prompt, two ranks
        _case("allreduce_512", "allreduce", 512, 1024, 1024, 2, 0, "fp16", False),
        # sequence-parallel input of a column-parallel projection, eight shards read in place
        _case("allgather_8x512", "allgather", 512, 4096, 1024, 8, 0, "bf16", False),
        # the same at a long prompt whose k is not a whole number of 16-byte pieces
        _case("allgather_8x1024_odd_k", "allgather", 1024, 6148, 5120, 8, 3, "fp16", False),
        # a prefill chunk on shards that fill no tile: 125 rows per rank, k = half a cache line over, biased, half output
        _case("quant_rs_chunk_1000", "quant_reduce_scatter", 1000, 1376, 4096, 8, 5, "fp16", True, bias=True, outbound=True),
        # a long W8A8 prefill as the benchmark runs it (checksums instead of stored tiles)
        _case("quant_rs_8192", "quant_reduce_scatter", 8192, 1792, 4096, 8, 0, "bf16", False),
        # the reference's own round structure: GEMM rounds, then int32 reduce rounds, on two streams
        _case("quant_pipelined_4096", "quant_pipelined", 4096, 1792, 4096, 8, 2, "bf16", False, int32_reduce=True, outbound=True),
        # ragged row blocks and columns (1018 rows per rank), weights stored output-major
        _case("rs_8144_ragged", "reduce_scatter", 8144, 5120, 1696, 8, 4, "fp16", True, outbound=True),
        # the largest: a long prefill through a down projection
        _case("rs_8192_long_k", "reduce_scatter", 8192, 27392, 4096, 8, 7, "fp16", True, outbound=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _whole(x, step, lo):
    return max(lo, int(round(x / step)) * step)


def draw(rng):
    op = rng.choice(["quant_decode", "quant_decode", "allreduce", "allreduce", "allgather", "quant_reduce_scatter",
                     "quant_reduce_scatter", "reduce_scatter", "quant_pipelined"])
    while True:
        ranks = rng.choice([2, 4, 8, 8])
        rank = rng.randrange(ranks)
        k = _whole(_log(rng, 512, 16384), rng.choice([256, 128, 128, 64, 64, 32, 4]), 128)
        n = _whole(_log(rng, 512, 8192), rng.choice([256, 256, 128, 128, 32]), 256)
        dtype = rng.choice(["fp16", "bf16"])
        trans_b = rng.random() < 0.6
        more = {}
        if op == "quant_decode":
            m = _log(rng, 1, 512)
            more = {"kept": rng.choice([m, -(-m // ranks)]), "bias": rng.random() < 0.3, "bound": rng.random() < 0.5}
        elif op == "allreduce":
            m = _log(rng, 1, 4096)
        elif op == "allgather":
            m = _log(rng, 1, 1024)
        elif op == "quant_pipelined":
            m = ranks * 128 * rng.randint(1, 32 // ranks)
            more = {"outbound": True, "int32_reduce": True}
        else:
            m = ranks * _log(rng, 8, 8192 // ranks)
            more = {"outbound": rng.random() < 0.7}
            if op == "quant_reduce_scatter":
                more.update({"bias": rng.random() < 0.3, "int32_reduce": rng.random() < 0.2, "bound": rng.random() < 0.5})
        rows = m * ranks if op == "allgather" else m
        if 2.0 * rows * k * n <= 6e11:
            return _case("", op, m, k, n, ranks, rank, dtype, trans_b, **more)


def _comm_type(op):
    return {"allreduce": lib.MATMUL_ALLREDUCE, "allgather": lib.ALLGATHER_MATMUL,
            "reduce_scatter": lib.MATMUL_REDUCE_SCATTER}.get(op, lib.QUANT_MATMUL_REDUCE_SCATTER)


def _tiling(case, comm, desc):
    """The library's own tiles, and as many tiles in one round as the call has, so that every tile has its own place in
    the symmetric workspace (a peer pulls them all after the call)."""
    pipelined = case["op"] == "quant_pipelined"
    t = ops.default_tiling(case["m"], case["k"], case["n"], case["ranks"], m0=128 if pipelined else 0, n0=256 if pipelined else 0, k0=0)
    tasks = int(lib.load().catcoc_get_task_count(comm, ctypes.byref(t), ctypes.byref(desc)))
    lib.check()
    t.commInterval = max(1, -(-tasks // 256))
    return t, tasks


def prepare(case, seed):
    m, k, n, P, rank, op = case["m"], case["k"], case["n"], case["ranks"], case["rank"], case["op"]
    tb, dt = case["trans_b"], _DT[case["dtype"]]
    g = torch.Generator(device=DEV).manual_seed(seed)
    comm = _comm_type(op)
    quant = op.startswith("quant")
    s = {"case": case}

    def normal(rows, cols, dtype, scale=1.0):
        t = torch.empty((rows, cols), dtype=dtype, device=DEV)
        return t.normal_(0.0, scale, generator=g)

    def int8(rows, cols):
        return torch.randint(-127, 128, (rows, cols), dtype=torch.int8, device=DEV, generator=g)

    wshape = (n, k) if tb else (k, n)
    kept = {"allreduce": m, "allgather": m * P, "quant_decode": case["kept"]}.get(op, m // P)
    if quant:
        s["a"], s["b"] = int8(m, k), int8(*wshape)
        s["scale_a"] = torch.empty(m, device=DEV).uniform_(0.005, 0.02, generator=g)
        s["scale_b"] = torch.empty(n, device=DEV).uniform_(0.001, 0.01, generator=g)
        s["bias"] = torch.randint(-1000, 1000, (n,), dtype=torch.int32, device=DEV, generator=g) if case["bias"] else None
    else:
        s["a"], s["b"] = normal(m, k, dt), normal(*wshape, dt, 0.02)
    if op == "allgather":
        s["peers"] = [normal(m, k, dt) for _ in range(P - 1)]
    elif case["int32_reduce"]:
        s["peers"] = [torch.randint(-2 ** 20, 2 ** 20, (kept, n), dtype=torch.int32, device=DEV, generator=g) for _ in range(P - 1)]
    else:
        s["peers"] = [normal(kept, n, torch.float32) for _ in range(P - 1)]
    s["out"] = torch.empty((kept, n), dtype=dt, device=DEV)
    s["outbound"] = s["checksum"] = None

    if op == "quant_decode":
        need = ops.splitk_plan(m, k, n, P, 0, kept)[0]
        s["workspace"] = torch.zeros(max(need, _COUNTERS), dtype=torch.uint8, device=DEV)
        if kept < m:   # the rows of the other ranks stay visible as sums
            s["checksum"] = torch.zeros(-(-m // 128) * -(-n // 128), dtype=torch.int64, device=DEV)
    else:
        desc = lib.make_desc(rank, P, [16] * (P - 1))
        t, tasks = _tiling(case, comm, desc)
        s["tiling"] = t
        if op in ("allreduce", "allgather", "reduce_scatter", "quant_reduce_scatter"):
            need = ops.kslice_plan(comm, lib.INT8 if quant else dt, m, k, n, rank, P, tiling=t)[0]
            s["workspace"] = torch.zeros(max(need, _COUNTERS), dtype=torch.uint8, device=DEV)
        if case["outbound"]:
            dtype_code = lib.INT8 if quant else (lib.FP16 if dt == torch.float16 else lib.BF16)
            size = int(lib.load().catcoc_get_workspace_size(comm, dtype_code, ctypes.byref(t), ctypes.byref(desc)))
            s["outbound"] = torch.zeros(size // 4, dtype=torch.int32 if case["int32_reduce"] else torch.float32, device=DEV)
        elif op == "quant_reduce_scatter":
            s["checksum"] = torch.zeros(tasks, dtype=torch.int64, device=DEV)
        elif op == "reduce_scatter":
            s["checksum"] = torch.zeros(tasks, dtype=torch.float64, device=DEV)
        if op == "quant_pipelined":
            s["sums"] = torch.empty((kept, n), dtype=torch.int32, device=DEV)
            s["stream"] = torch.cuda.Stream()
            s["plan"] = ops.PipelinedPlan(ops.pipelined_round_count(comm, t, rank, P))
    if case["bound"]:
        s["launch"] = _bind(s)
    return s


def _quant_arguments(s):
    c = s["case"]
    a = (s["a"], s["b"], s["scale_a"], s["scale_b"], s["bias"], s["peers"])
    if c["op"] == "quant_decode":
        return a, dict(rank_size=c["ranks"], kept_row_begin=0, kept_rows=c["kept"], workspace=s["workspace"], checksum=s["checksum"],
                       out=s["out"], trans_b=c["trans_b"], reduce_int32=c["int32_reduce"])
    return a, dict(rank=c["rank"], rank_size=c["ranks"], tiling=s["tiling"], trans_b=c["trans_b"], reduce_int32=c["int32_reduce"],
                   outbound=s["outbound"], checksum=s["checksum"], out=s["out"], workspace=s["workspace"])


def _bind(s):
    a, kw = _quant_arguments(s)
    make = ops.prepare_quant_matmul_splitk if s["case"]["op"] == "quant_decode" else ops.prepare_quant_matmul_reduce_scatter
    return make(*a, **kw)[0]


def run(s):
    c = s["case"]
    op, P, rank, tb = c["op"], c["ranks"], c["rank"], c["trans_b"]
    if c["bound"]:
        s["launch"]()
    elif op == "quant_decode":
        a, kw = _quant_arguments(s)
        ops.quant_matmul_splitk(*a, **kw)
    elif op == "quant_reduce_scatter":
        a, kw = _quant_arguments(s)
        ops.quant_matmul_reduce_scatter(*a, **kw)
    elif op == "quant_pipelined":
        ops.pipelined_quant_matmul_reduce_scatter(s["a"], s["b"], s["scale_a"], s["scale_b"], s["bias"], s["peers"], rank, P, s["outbound"],
                                                  c_accum=s["sums"], tiling=s["tiling"], trans_b=tb, comm_stream=s["stream"], out=s["out"],
                                                  plan=s["plan"])
        return {"out": s["out"], "sums": s["sums"], "outbound": s["outbound"]}
    elif op == "allreduce":
        ops.matmul_allreduce(s["a"], s["b"], s["peers"], rank, P, tiling=s["tiling"], trans_b=tb, out=s["out"], workspace=s["workspace"])
    elif op == "allgather":
        ops.allgather_matmul(s["a"], s["peers"], s["b"], rank, P, tiling=s["tiling"], trans_b=tb, out=s["out"], workspace=s["workspace"])
    else:
        ops.matmul_reduce_scatter(s["a"], s["b"], s["peers"], rank, P, tiling=s["tiling"], trans_b=tb, outbound=s["outbound"],
                                  checksum=s["checksum"], out=s["out"], workspace=s["workspace"])
    return {key: s[key] for key in ("out", "outbound", "checksum") if s[key] is not None}


def work(case):
    m, k, n, P, op = case["m"], case["k"], case["n"], case["ranks"], case["op"]
    es = 1 if op.startswith("quant") else 2
    rows = m * P if op == "allgather" else m
    kept = {"allreduce": m, "allgather": rows, "quant_decode": case["kept"]}.get(op, m // P)
    moved = (rows * k + k * n) * es + kept * n * 2
    if es == 1:
        moved += 4 * (m + n) + (4 * n if case["bias"] else 0)
    if op != "allgather":
        moved += (P - 1) * kept * n * 4
    if case["outbound"]:
        moved += (m - kept) * n * 4
    if op == "quant_pipelined":
        moved += kept * n * 4   # the int32 sums are an output too
    return {"bytes": moved, "flops": 2 * rows * k * n}


def tolerance(case):
    # The integer part of the W8A8 operators (checksums, int32 sums, int32 tiles) has one right answer.  What remains is the
    # order of 32-bit float sums in front of one rounding to 16 bits: a last-place change in a few outputs.  Against the same
    # sums in 64 bits the outputs here are off by up to 1e-4 (bf16) / 3e-5 (fp16) in the 2-norm and by one last place (2^-7 /
    # 2^-10 of the value) at most; k = 27392 sums a little further.
    if case["op"] == "quant_pipelined":
        return "exact"
    return {"rel": 4e-4, "max": 3e-2} if case["dtype"] == "bf16" else {"rel": 2e-4, "max": 4e-3}
