"""The compiled operator call (csrc/host_call.cpp) against the Python path it stands in front of: the same outputs where it takes a call, the same error where
neither does."""
import pytest
import torch

from mm_rs_with_catlass_amd import lib as L
from mm_rs_with_catlass_amd import ops
from test_gpu_parity import _need_gpu

pytestmark = pytest.mark.gpu
M, K, N, P = 48, 160, 272, 4


def arguments(op, **change):
    """One call of every kind, all optional operands in it; `change` replaces operands by what f(operand) returns."""
    g = torch.Generator(device="cuda:0").manual_seed(3)
    f = lambda *s: torch.randn(s, device="cuda:0", generator=g)
    i8 = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device="cuda:0", generator=g)
    ws = torch.zeros(1 << 20, dtype=torch.uint8, device="cuda:0")
    kw = dict(rank_size=P, trans_b=True, workspace=ws, out=None)
    if op in ("allreduce", "allgather", "reduce_scatter"):
        kw.update(a=f(M, K).bfloat16(), b=f(N, K).bfloat16(), rank=1)
        rows = {"allreduce": M, "allgather": M * P, "reduce_scatter": M // P}[op]
        kw["acc_dump"] = torch.zeros(M * P if op == "allgather" else M, N, device="cuda:0")
        if op == "allgather":
            kw["a_local"] = kw.pop("a")
            kw["peer_shards"] = [f(M, K).bfloat16() for _ in range(P - 1)]
        else:
            kw.update(peers=[f(rows + 3, N + 8) for _ in range(P - 1)], peer_row_offset=2)
        if op == "reduce_scatter":
            kw.update(outbound=torch.zeros(256 * 2 * 64 * 256, device="cuda:0"))
    else:
        kw.update(x1=i8(M, K), x2=i8(N, K), scale_x1=f(M).abs(), scale_x2=f(N).abs(), bias=torch.arange(N, dtype=torch.int32, device="cuda:0"), out_dtype=torch.float16)
        rows = 10 if op == "quant_decode" else M // P
        kw.update(peers=tuple(f(rows, N) for _ in range(P - 1)), c_accum=torch.zeros(rows, N, dtype=torch.int32, device="cuda:0"))
        kw["checksum"] = torch.zeros(64, dtype=torch.int64, device="cuda:0")
        kw.update(dict(kept_row_begin=5, kept_rows=10) if op == "quant_decode" else dict(rank=2))
    for key, how in change.items():
        kw[key] = how(kw[key]) if callable(how) else how
    return kw


CALLS = {"allreduce": ops.matmul_allreduce, "allgather": ops.allgather_matmul, "reduce_scatter": ops.matmul_reduce_scatter,
         "quant_reduce_scatter": ops.quant_matmul_reduce_scatter, "quant_decode": ops.quant_matmul_splitk}


def both(monkeypatch, op, **change):
    """[(output and what else was written, or the error's text)] of the two paths, and whether the compiled one took the call."""
    native, took, results = L.load_host().call, [], []

    def first(*a):
        out = native(*a)
        took.append(out is not None)
        return out

    for call in (first, lambda *a: None):
        monkeypatch.setattr(ops, "_call", call)
        kw = arguments(op, **change)
        try:
            out = CALLS[op](**kw)
            torch.cuda.synchronize()
            results.append([out] + [kw[k] for k in ("acc_dump", "outbound", "checksum", "c_accum") if kw.get(k) is not None])
        except (L.CatcocError, TypeError, AttributeError) as e:
            results.append((type(e), str(e)))
    return results[0], results[1], took == [True]


@pytest.mark.parametrize("op", list(CALLS))
@pytest.mark.parametrize("change", [{}, {"out": "given"}, {"tiling": "given"}, {"swizzle": (3, 0)}, {"workspace": None}, {"block_num": 128}])
def test_takes_the_ordinary_call(op, change, monkeypatch):
    _need_gpu()
    change = dict(change)
    rows = {"allreduce": M, "allgather": M * P, "quant_decode": 10}.get(op, M // P)
    if "out" in change:
        change["out"] = torch.zeros(rows, N, dtype=torch.float16 if op.startswith("quant") else torch.bfloat16, device="cuda:0")
    if "tiling" in change:
        if op == "quant_decode":
            pytest.skip("takes no tiling")
        change["tiling"] = ops.default_tiling(M, K, N, P, m0=0, n0=0, k0=0)
    a, b, took = both(monkeypatch, op, **change)
    assert took and not isinstance(a, tuple), a
    assert len(a) == len(b) and all(x.dtype == y.dtype and torch.equal(x, y) for x, y in zip(a, b))


# (what an operator does not have is not there to be wrong)
@pytest.mark.parametrize("op,name", [(op, name) for op in CALLS for name in ["a", "b", "peers", "out", "workspace", "rank_size", "scale", "dump", "tiling", "trans", "subclass", "checksum", "host"]
                                     if (op, name) not in [("quant_decode", "tiling"), ("allreduce", "checksum"), ("allgather", "checksum")] and (op.startswith("quant") or name != "scale")])
def test_leaves_the_others_to_the_python_path(op, name, monkeypatch):
    _need_gpu()
    quant = op.startswith("quant")
    first, second = ("x1", "x2") if quant else ("a_local" if op == "allgather" else "a", "b")
    peers = "peer_shards" if op == "allgather" else "peers"

    class Sub(torch.Tensor):
        pass

    sums = lambda count, dtype: {"outbound": None, "checksum": torch.zeros(count, dtype=dtype, device="cuda:0")}
    changes = {
        "a": [{first: lambda t: t[:, ::2]}, {first: lambda t: t.float()}, {first: lambda t: t[0]}, {first: lambda t: t.t()}],
        "b": [{second: lambda t: t[:, :-1].contiguous()}, {second: lambda t: t.float()}],
        "peers": [{peers: lambda p: p[:-1]}, {peers: lambda p: [t[:5] for t in p]}, {peers: lambda p: [t[:, :-16].contiguous() for t in p]}, {peers: lambda p: [t.double() for t in p]},
                  {peers: lambda p: [p[0][:, :-1].contiguous()] + list(p[1:])}],
        "out": [{"out": torch.zeros(3, N, dtype=torch.bfloat16, device="cuda:0")}, {"out": torch.zeros(M, N, device="cuda:0")}],
        "workspace": [{"workspace": lambda t: t.cpu()}],
        "rank_size": [{"rank_size": 17}, {"rank_size": 0}, {"rank_size": -4}],
        "scale": [{"scale_x1": lambda t: t[:-1]}, {"scale_x2": lambda t: t.double()}, {"bias": lambda t: t[:5]}, {"c_accum": lambda t: t[0]}],
        "dump": [{"acc_dump": torch.zeros(5, dtype=torch.int32 if quant else torch.float32, device="cuda:0")}],
        "tiling": [{"tiling": ops.default_tiling(M + P, K, N, P)}, {"tiling": bytes(48)}, {"tiling": ops.default_tiling(M, K, N, P, rankSize=P + 1)}],
        "trans": [{"trans_b": False}, {"peer_row_offset": -1}] if op != "allgather" else [{"trans_b": False}],
        "subclass": [{first: lambda t: t.as_subclass(Sub)}],
        "checksum": [{"checksum": torch.zeros(1, dtype=torch.int32, device="cuda:0")}, {"checksum": torch.zeros(0, dtype=torch.int64, device="cuda:0")}] if quant else
                    [sums(64, torch.float32), sums(64, torch.int64), sums(1, torch.float64)],
        "host": [{first: lambda t: t.cpu()}, {peers: lambda p: [t.cpu() for t in p]}],
    }[name]
    assert changes
    for change in changes:
        a, b, took = both(monkeypatch, op, **change)
        assert not took, change
        if isinstance(a, tuple):
            assert a == b
        else:
            assert all(torch.equal(x, y) for x, y in zip(a, b))
