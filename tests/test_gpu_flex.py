"""GPU parity of launches in flexible mode (csrc/gemm_flex.h): row tiles over the rows of all ranks wherever the ranks'
boundaries lie, k and n that fill no step and no tile.  Bars as in test_gpu_parity: int32 accumulators, checksums and W8A8
outputs bit for bit, workspace tiles bit for bit, float outputs within the reference's gate."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle
from mm_rs_with_catlass_amd import lib as L
from mm_rs_with_catlass_amd import ops
from test_gpu_parity import TORCH_DT, _check_float, _need_gpu, _rand16, dev, dev16, host16, quant_case

pytestmark = pytest.mark.gpu


def peers_of(rng, M, N, K, P, rank, ri):
    """The peers quant_case draws from the same generator (after operands, scales and bias)."""
    rng.integers(-127, 128, (M, K), dtype=np.int8)
    rng.integers(-127, 128, (K, N), dtype=np.int8)
    rng.uniform(0.005, 0.02, M), rng.uniform(0.001, 0.01, N), rng.integers(-1000, 1000, N, dtype=np.int32)
    rows = M // P
    if ri:
        return [rng.integers(-2 ** 24, 2 ** 24, (rows, N), dtype=np.int32) for _ in range(P - 1)]
    return [rng.standard_normal((rows, N)).astype(np.float32) for _ in range(P - 1)]


def sum_bound(A, B, dtype):
    """How far two fp32 sums of the same K products may be apart, per element: each is within 4 sqrt(K) 2^-24 |a||b| of the exact
    sum (roundings of K additions that are independent, four standard deviations; sum |a_i b_i| <= |a||b|).  At K = 6148 that
    is a tenth of what four products more or less make."""
    a, b = oracle.half_to_f32(A, dtype), oracle.half_to_f32(B, dtype)
    return 8 * np.sqrt(A.shape[1]) * 2.0 ** -24 * np.outer(np.linalg.norm(a, axis=1), np.linalg.norm(b, axis=0)) + 1e-9


def tasks_of(comm, t, d):
    """(task, target rank, first row, first column, workspace row) of every task of a launch."""
    tr, row, col, ws = (C.c_uint32() for _ in range(4))
    for task in range(L.load().catcoc_get_task_count(comm, C.byref(t), C.byref(d))):
        L.load().catcoc_task_tile(comm, C.byref(t), C.byref(d), task, C.byref(tr), C.byref(row), C.byref(col), C.byref(ws))
        yield task, tr.value, row.value, col.value, ws.value


# (rows per rank, N, K, P, rank, weights as [n,k], int32 peers, m0, commInterval)
@pytest.mark.parametrize("outbound", [False, True])
@pytest.mark.parametrize("case", [(125, 512, 1376, 8, 5, True, False, 0, 1),     # one rank per tile; half a step of k left
                                  (1, 260, 68, 16, 15, False, False, 0, 1),      # 16 tasks in one tile, rows of B end inside a 16-byte piece
                                  (8, 256, 64, 8, 0, False, True, 0, 1),         # whole steps of k, raw int32 tiles
                                  (9, 36, 4, 4, 1, True, False, 0, 1),           # no whole step of k at all
                                  (63, 1028, 192, 4, 2, False, False, 0, 1),     # whole k, but B's last step is checked (N % 16)
                                  (65, 772, 260, 8, 7, True, True, 0, 1),        # tiles straddle ranks
                                  (200, 300, 320, 2, 1, False, False, 64, 2),    # caller's 64-row tiles, several per rank, two rounds
                                  (300, 516, 100, 4, 3, True, False, 0, 1)])     # more than one tile per rank
def test_quant_rs_any_rows_any_k(case, outbound):
    rows, N, K, P, rank, tb, ri, m0, ci = case
    M = rows * P
    t = ops.default_tiling(M, K, N, P, m0=m0, n0=0, k0=0, commInterval=ci)
    bn = 16 if ci > 1 else 0
    r = quant_case(np.random.default_rng(rows), M, N, K, P, rank, bias=True, trans_b=tb, reduce_int32=ri, tiling=t, outbound=outbound,
                   launches=2, block_num=bn)
    assert r["exact"] == r["total"]
    # the same in k slices (a second launch adds them up); the counter block of the workspace stays zero
    if K >= 128:
        g = lambda a: None if a is None else dev(a)
        ws = torch.zeros(65536 + 3 * M * N * 4, dtype=torch.uint8, device="cuda:0")
        ws[65536:] = 0x55
        peers = peers_of(np.random.default_rng(rows), M, N, K, P, rank, ri)
        kw = {"outbound": torch.zeros_like(r["outbound"])} if outbound else {"checksum": torch.full_like(r["checksum"], 77)}
        out = ops.quant_matmul_reduce_scatter(dev(r["x1"]), dev(np.ascontiguousarray(r["x2"].T) if tb else r["x2"]), dev(r["s1"]), dev(r["s2"]),
                                              g(r["bias"]), [dev(p) for p in peers], rank, P, tiling=t, trans_b=tb, reduce_int32=ri,
                                              block_num=bn, workspace=ws, split_k=3, **kw)
        torch.cuda.synchronize()
        assert np.array_equal(host16(out), r["out_want"]) and not ws[:65536].any() and bool((ws[65536:] != 0x55).any())
        if outbound:
            assert torch.equal(kw["outbound"].view(torch.int32), r["outbound"].view(torch.int32))
        else:
            others = r["checksum"] != 0
            assert torch.equal(kw["checksum"][others], r["checksum"][others])
    d = L.make_desc(rank, P, [16] * (P - 1), block_num=bn)
    tr, row, col, ws = (C.c_uint32() for _ in range(4))
    step = m0 or (64 if rows <= 64 else 128)
    deq = r["acc"] if ri else oracle.dequant(r["acc"], r["s2"], r["s1"])
    for task in range(r["ntasks"]):
        L.load().catcoc_task_tile(L.QUANT_MATMUL_REDUCE_SCATTER, C.byref(t), C.byref(d), task, C.byref(tr), C.byref(row), C.byref(col), C.byref(ws))
        if tr.value == rank:
            continue
        r1, c1 = min(row.value + step, (tr.value + 1) * rows), min(col.value + 256, N)
        if outbound:
            got = r["outbound"].cpu().numpy().reshape(-1, 256)[ws.value:ws.value + r1 - row.value, :c1 - col.value]
            want = deq[row.value:r1, col.value:c1]
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), task
        else:
            assert int(r["checksum"][task]) == int(r["acc"][row.value:r1, col.value:c1].astype(np.int64).sum()), task


# (op, rows (of a shard for all-gather), N, K, P, weights as [n,k])
@pytest.mark.parametrize("dtype", [oracle.FP16, oracle.BF16])
@pytest.mark.parametrize("case", [("allreduce", 1, 256, 128, 8, True), ("allreduce", 33, 516, 1000, 4, False), ("allreduce", 129, 260, 66, 2, False),
                                  ("allgather", 3, 264, 516, 8, True), ("allgather", 65, 768, 1026, 4, False), ("allgather", 200, 1284, 6148, 2, False)])
def test_float_any_rows_any_k(dtype, case):
    _need_gpu()
    op, m, N, K, P, tb = case
    rng = np.random.default_rng(m + K)
    B = _rand16(rng, (K, N), dtype, 0.02)
    Bd = dev16(np.ascontiguousarray(B.T) if tb else B, dtype)
    rank = P - 1
    if op == "allgather":
        shards = [_rand16(rng, (m, K), dtype) for _ in range(P)]
        ds = [dev16(s, dtype) for s in shards]
        dump = torch.zeros((m * P, N), dtype=torch.float32, device="cuda:0")
        out = ops.allgather_matmul(ds[rank], ds[:rank], Bd, rank, P, trans_b=tb, acc_dump=dump)
        torch.cuda.synchronize()
        part = oracle.gemm_half_f32(np.concatenate(shards, 0), B, dtype)
        full, want = part, oracle.allgather_matmul(shards, B, dtype)
    else:
        A = _rand16(rng, (m, K), dtype)
        peers = [rng.standard_normal((m, N)).astype(np.float32) for _ in range(P - 1)]
        part, want = oracle.matmul_reduce(A, B, dtype, 0, m, peers, want_partial=True)
        full = part + sum(peers)
        dump = torch.zeros((m, N), dtype=torch.float32, device="cuda:0")
        out = ops.matmul_allreduce(dev16(A, dtype), Bd, [dev(p) for p in peers], rank, P, trans_b=tb, acc_dump=dump)
        torch.cuda.synchronize()
    _check_float(host16(out), want, full, dtype, K)
    assert out.dtype == TORCH_DT[dtype]
    if K >= 512:   # in k slices: added in slice order, so twice the same bits
        ws = torch.zeros(65536 + 5 * out.numel() * 4, dtype=torch.uint8, device="cuda:0")
        again = []
        for _ in range(2):
            if op == "allgather":
                o = ops.allgather_matmul(ds[rank], ds[:rank], Bd, rank, P, trans_b=tb, workspace=ws, split_k=5)
            else:
                o = ops.matmul_allreduce(dev16(A, dtype), Bd, [dev(p) for p in peers], rank, P, trans_b=tb, workspace=ws, split_k=5)
            torch.cuda.synchronize()
            again.append(host16(o))
        assert np.array_equal(again[0], again[1])
        _check_float(again[0], want, full, dtype, K)
    assert (np.abs(dump.cpu().numpy() - part) <= sum_bound(np.concatenate(shards, 0) if op == "allgather" else A, B, dtype)).all()


@pytest.mark.parametrize("dtype", [oracle.FP16, oracle.BF16])
def test_float_reduce_scatter_checksums_of_small_ranks(dtype):
    """Several tasks in one tile: each one's sum, and the kept block with its peers."""
    _need_gpu()
    P, rows, N, K, rank = 8, 11, 300, 200, 3
    rng = np.random.default_rng(31)
    A, B = _rand16(rng, (P * rows, K), dtype), _rand16(rng, (K, N), dtype, 0.02)
    peers = [rng.standard_normal((rows, N)).astype(np.float32) for _ in range(P - 1)]
    part, want = oracle.matmul_reduce(A, B, dtype, rank * rows, rows, peers, want_partial=True)
    cs = torch.zeros(2 * P, dtype=torch.float64, device="cuda:0")
    out = ops.matmul_reduce_scatter(dev16(A, dtype), dev16(B, dtype), [dev(p) for p in peers], rank, P, checksum=cs)
    torch.cuda.synchronize()
    _check_float(host16(out), want, part[rank * rows:(rank + 1) * rows] + sum(peers), dtype, K)
    t = ops.default_tiling(P * rows, K, N, P, m0=0, n0=0, k0=0)
    d = L.make_desc(rank, P, [16] * (P - 1))
    bounds = sum_bound(A, B, dtype)
    tr, row, col = C.c_uint32(), C.c_uint32(), C.c_uint32()
    for task in range(2 * P):
        L.load().catcoc_task_tile(L.MATMUL_REDUCE_SCATTER, C.byref(t), C.byref(d), task, C.byref(tr), C.byref(row), C.byref(col), None)
        at = np.s_[row.value:row.value + rows, col.value:min(col.value + 256, N)]
        blk = part[at].astype(np.float64)
        assert abs(float(cs[task]) - (0.0 if tr.value == rank else blk.sum())) <= bounds[at].sum(), task


# (m, N, K, P, kept rows [begin, +count), weights as [n,k], int32 peers): kept rows that start, end or lie inside a 64-row tile,
# a last row tile and a last 128-column block of their own, at most 32 rows with a long k, every row kept
@pytest.mark.parametrize("case", [(65, 384, 512, 4, 63, 2, False, False), (130, 1152, 1024, 8, 60, 11, True, True), (200, 256, 448, 2, 64, 64, False, False),
                                  (511, 640, 1792, 8, 510, 1, True, False), (5, 128, 4096, 8, 1, 2, False, True), (32, 512, 8192, 1, 0, 4, False, False),
                                  (33, 128, 192, 2, 0, 33, True, False), (256, 512, 2048, 8, 0, 256, False, True), (384, 1024, 512, 4, 32, 96, True, False)])
def test_quant_kept_rows_in_slices(case):
    """Explicit kept rows in k slices: partial sums of the kept rows only, the other rows as sums per slice."""
    _need_gpu()
    M, N, K, P, kb, kr, tb, ri = case
    rng = np.random.default_rng(M + N)
    x1, x2 = rng.integers(-127, 128, (M, K), dtype=np.int8), rng.integers(-127, 128, (K, N), dtype=np.int8)
    s1, s2 = rng.uniform(0.005, 0.02, M).astype(np.float32), rng.uniform(0.001, 0.01, N).astype(np.float32)
    b = rng.integers(-1000, 1000, N, dtype=np.int32)
    peers = [rng.integers(-2 ** 24, 2 ** 24, (kr, N), dtype=np.int32) if ri else rng.standard_normal((kr, N)).astype(np.float32) for _ in range(P - 1)]
    acc, want = oracle.quant_matmul_reduce_scatter(x1, x2, s1, s2, b, kb, kr, peers, oracle.BF16, reduce_int32=ri)
    need, _, tiles = ops.splitk_plan(M, K, N, P, kb, kr)
    sums = np.array([[acc[r:r + 128, c:c + 128].astype(np.int64).sum() - acc[max(r, kb):max(min(r + 128, kb + kr), max(r, kb)), c:c + 128].astype(np.int64).sum()
                      for c in range(0, N, 128)] for r in range(0, M, 128)]).ravel()
    x2d = dev(np.ascontiguousarray(x2.T) if tb else x2)
    for extra in (0, 1 << 20):   # the query's workspace, and a larger one, whose rest stays as it was
        ws = torch.zeros(max(need, 65536) + extra, dtype=torch.uint8, device="cuda:0")
        ws[65536:] = 0x55
        cs = torch.full((tiles,), -7, dtype=torch.int64, device="cuda:0") if kr < M else None
        ca = torch.full((kr, N), -7, dtype=torch.int32, device="cuda:0")
        out = ops.quant_matmul_splitk(dev(x1), x2d, dev(s1), dev(s2), dev(b), [dev(p) for p in peers], P, kb, kr, workspace=ws, checksum=cs,
                                      c_accum=ca, trans_b=tb, reduce_int32=ri)
        torch.cuda.synchronize()
        assert np.array_equal(host16(out), want) and not ws[:65536].any()
        assert need == 0 or K < 512 or bool((ws[65536:need] != 0x55).any())   # (slices did run; eight k steps make two of them)
        assert bool((ws[max(need, 65536):] == 0x55).all())
        assert np.array_equal(ca.cpu().numpy(), acc[kb:kb + kr] + (sum(peers) if ri else 0))
        if cs is not None:
            assert np.array_equal(cs.cpu().numpy(), sums)


@pytest.mark.parametrize("case", [(257, 512, 4096, 8), (256, 256, 8192, 2), (131, 300, 2048, 4), (448, 3584, 8224, 2)])
def test_float_allreduce_few_tiles_long_k(case):
    """All-reduce launches whose workspace query asks for the flexible tiles' own slices: with that workspace, with less (the
    slices that fit) and with none; aligned and ragged rows, two workgroups per CU (98 tiles)."""
    _need_gpu()
    M, N, K, P = case
    rng = np.random.default_rng(M)
    A, B = _rand16(rng, (M, K), oracle.BF16), _rand16(rng, (K, N), oracle.BF16, 0.02)
    peers = [rng.standard_normal((M, N)).astype(np.float32) for _ in range(P - 1)]
    part, want = oracle.matmul_reduce(A, B, oracle.BF16, 0, M, peers, want_partial=True)
    need, f = ops.kslice_plan(L.MATMUL_ALLREDUCE, torch.bfloat16, M, K, N, 0, P)
    assert need >= 65536 + 4 * M * N * 4 and (f == 2) == (M % 128 == 0)   # (an aligned launch's count is the aligned kernel's)
    for size in (need, 65536 + 2 * M * N * 4 + 4096, 0):
        ws = torch.zeros(size, dtype=torch.uint8, device="cuda:0") if size else None
        if ws is not None:
            ws[65536:] = 0x55
        try:
            out = ops.matmul_allreduce(dev16(A, oracle.BF16), dev16(B, oracle.BF16), [dev(p) for p in peers], P - 1, P, workspace=ws)
        except L.CatcocError as e:   # (the aligned kernel's own two slices are the least an aligned launch takes with a workspace)
            assert 0 < size < need and "workspace too small" in str(e) and M % 128 == 0
            continue
        torch.cuda.synchronize()
        _check_float(host16(out), want, part + sum(peers), oracle.BF16, K)
        assert ws is None or not ws[:65536].any()


def test_float_reduce_scatter_ragged_few_tiles_long_k():
    """Reduce-scatter with stored tiles on ragged rows: k slices in the workspace the query asks for, and whole tiles without it."""
    _need_gpu()
    P, rows, N, K, rank = 4, 150, 296, 4096, 2
    M = P * rows
    rng = np.random.default_rng(77)
    A, B = _rand16(rng, (M, K), oracle.FP16), _rand16(rng, (K, N), oracle.FP16, 0.02)
    peers = [rng.standard_normal((rows, N)).astype(np.float32) for _ in range(P - 1)]
    part, want = oracle.matmul_reduce(A, B, oracle.FP16, rank * rows, rows, peers, want_partial=True)
    t = ops.default_tiling(M, K, N, P, m0=0, n0=0, k0=0)
    need, f = ops.kslice_plan(L.MATMUL_REDUCE_SCATTER, torch.float16, M, K, N, rank, P, tiling=t)
    assert f >= 4 and need == 65536 + f * M * N * 4
    d = L.make_desc(rank, P, [16] * (P - 1))
    tr, row, col, wsr = (C.c_uint32() for _ in range(4))
    tasks = L.load().catcoc_get_task_count(L.MATMUL_REDUCE_SCATTER, C.byref(t), C.byref(d))
    size = L.load().catcoc_get_workspace_size(L.MATMUL_REDUCE_SCATTER, L.FP16, C.byref(t), C.byref(d))
    bounds = sum_bound(A, B, oracle.FP16)
    for ws in (torch.zeros(need, dtype=torch.uint8, device="cuda:0"), None):
        ob = torch.full((size // 4,), 3.0, dtype=torch.float32, device="cuda:0")
        out = ops.matmul_reduce_scatter(dev16(A, oracle.FP16), dev16(np.ascontiguousarray(B.T), oracle.FP16), [dev(p) for p in peers], rank, P, tiling=t,
                                        trans_b=True, outbound=ob, workspace=ws)
        torch.cuda.synchronize()
        _check_float(host16(out), want, part[rank * rows:(rank + 1) * rows] + sum(peers), oracle.FP16, K)
        for task in range(tasks):
            L.load().catcoc_task_tile(L.MATMUL_REDUCE_SCATTER, C.byref(t), C.byref(d), task, C.byref(tr), C.byref(row), C.byref(col), C.byref(wsr))
            if tr.value == rank:
                continue
            r1, c1 = min(row.value + 128, (tr.value + 1) * rows), min(col.value + 256, N)
            got = ob.cpu().numpy().reshape(-1, 256)[wsr.value:wsr.value + r1 - row.value, :c1 - col.value]
            assert (np.abs(got - part[row.value:r1, col.value:c1]) <= bounds[row.value:r1, col.value:c1]).all(), task


# (rows per rank, N, K, P, rank, weights as [n,k]): one-round pipelined calls on ragged columns, ragged rows, and few aligned tiles: all on small tiles
@pytest.mark.parametrize("case", [(128, 640, 448, 8, 3, False), (256, 1440, 192, 4, 0, True), (72, 288, 100, 2, 1, False), (128, 512, 1792, 8, 7, True)])
@pytest.mark.parametrize("deterministic", [True, False])
def test_pipelined_quant_one_round(case, deterministic, kernel=L.KERNEL_SMALL):
    _need_gpu()
    rows, N, K, P, rank, tb = case
    M = rows * P
    rng = np.random.default_rng(rows + N)
    x1, x2 = rng.integers(-127, 128, (M, K), dtype=np.int8), rng.integers(-127, 128, (K, N), dtype=np.int8)
    s1, s2 = rng.uniform(0.005, 0.02, M).astype(np.float32), rng.uniform(0.001, 0.01, N).astype(np.float32)
    b = rng.integers(-1000, 1000, N, dtype=np.int32)
    peers = [rng.integers(-2 ** 20, 2 ** 20, (rows, N), dtype=np.int32) for _ in range(P - 1)]
    acc, want = oracle.quant_matmul_reduce_scatter(x1, x2, s1, s2, b, rank * rows, rows, peers, oracle.BF16, reduce_int32=True)
    t = ops.default_tiling(M, K, N, P, m0=128, n0=256, k0=0, commInterval=max(1, -(-(P * -(-rows // 128) * -(-N // 256)) // 256)))
    d = L.make_desc(rank, P, [16] * (P - 1))
    size = L.load().catcoc_get_workspace_size(L.QUANT_MATMUL_REDUCE_SCATTER, L.INT8, C.byref(t), C.byref(d))
    assert ops.pipelined_round_count(L.QUANT_MATMUL_REDUCE_SCATTER, t, rank, P) == 1
    ob = torch.full((size // 4,), -9, dtype=torch.int32, device="cuda:0")
    out, sums = ops.pipelined_quant_matmul_reduce_scatter(dev(x1), dev(np.ascontiguousarray(x2.T) if tb else x2), dev(s1), dev(s2), dev(b), [dev(p) for p in peers],
                                                          rank, P, ob, tiling=t, trans_b=tb, deterministic=deterministic)
    assert L.last_launch().kernel == kernel
    torch.cuda.synchronize()
    assert np.array_equal(sums.cpu().numpy(), acc[rank * rows:(rank + 1) * rows] + sum(peers)) and np.array_equal(host16(out), want)
    tr, row, col, wsr = (C.c_uint32() for _ in range(4))
    tiles = ob.cpu().numpy().reshape(-1, 256)
    for task in range(L.load().catcoc_get_task_count(L.QUANT_MATMUL_REDUCE_SCATTER, C.byref(t), C.byref(d))):
        L.load().catcoc_task_tile(L.QUANT_MATMUL_REDUCE_SCATTER, C.byref(t), C.byref(d), task, C.byref(tr), C.byref(row), C.byref(col), C.byref(wsr))
        if tr.value != rank:
            r1, c1 = min(row.value + 128, (tr.value + 1) * rows), min(col.value + 256, N)
            got = tiles[wsr.value:wsr.value + r1 - row.value, :c1 - col.value]
            assert np.array_equal(got, acc[row.value:r1, col.value:c1]), task


# one-round pipelined calls of whole tiles: few of them, on small ones; on aligned ones, whose peers the GEMM launch adds (two ranks, four with a short k, few
# tiles, more than there are CUs); and one that keeps its comm launch
@pytest.mark.parametrize("case", [(128, 512, 576, 2, 1, True), (256, 256, 960, 2, 0, False), (128, 512, 64, 4, 2, False), (128, 512, 960, 8, 6, True), (256, 3072, 512, 8, 4, True),
                                  (384, 1536, 576, 4, 1, False), (384, 3072, 576, 2, 0, True), (512, 3072, 576, 8, 7, False), (384, 4096, 448, 8, 3, True)])
@pytest.mark.parametrize("deterministic", [True, False])
def test_pipelined_quant_one_round_on_aligned_tiles(case, deterministic):
    rows, N, K, P, _, _ = case
    test_pipelined_quant_one_round(case, deterministic, L.KERNEL_ALIGNED if rows * P * N >= 48 * 128 * 256 else L.KERNEL_SMALL)


# kept tiles as halves in one round of workgroups, faster than mixed tiles
@pytest.mark.parametrize("case", [(512, 3072, 1280, 8, 2, False), (512, 3072, 1280, 8, 5, True)])
def test_pipelined_quant_one_round_with_halves(case):
    test_pipelined_quant_one_round(case, True, L.KERNEL_ALIGNED)


# one-round pipelined calls that one launch of small tiles takes: 128 and 64 rows by 128 columns, 32 and 64 rows by 64, ranks of ragged rows
@pytest.mark.parametrize("case", [(512, 2048, 1664, 4, 1, True), (128, 1408, 1504, 8, 6, True), (61, 1540, 1236, 8, 2, True), (96, 1040, 1280, 8, 0, False), (384, 1024, 1028, 2, 1, True)])
def test_pipelined_quant_one_round_on_small_tiles(case):
    test_pipelined_quant_one_round(case, True)


@pytest.mark.parametrize("tb", [False, True])
def test_pipelined_quant_one_round_equals_two(tb):
    """384 tiles: one round (the GEMM launch adds the peers) against two rounds with comm launches."""
    _need_gpu()
    M, N, K, P, rank = 1024, 12288, 64, 8, 5
    rows = M // P
    g = torch.Generator(device="cuda:0").manual_seed(11)
    x1, x2 = (torch.randint(-127, 128, s, dtype=torch.int8, device="cuda:0", generator=g) for s in ((M, K), (N, K) if tb else (K, N)))
    s1, s2 = (torch.empty(c, device="cuda:0").uniform_(0.001, 0.02, generator=g) for c in (M, N))
    peers = [torch.randint(-2 ** 20, 2 ** 20, (rows, N), dtype=torch.int32, device="cuda:0", generator=g) for _ in range(P - 1)]
    got = []
    for interval in (2, 1):
        t = ops.default_tiling(M, K, N, P, m0=128, n0=256, k0=0, commInterval=interval)
        assert ops.pipelined_round_count(L.QUANT_MATMUL_REDUCE_SCATTER, t, rank, P) == 3 - interval
        d = L.make_desc(rank, P, [16] * (P - 1))
        size = L.load().catcoc_get_workspace_size(L.QUANT_MATMUL_REDUCE_SCATTER, L.INT8, C.byref(t), C.byref(d))
        ob = torch.zeros(size // 4, dtype=torch.int32, device="cuda:0")
        got.append(ops.pipelined_quant_matmul_reduce_scatter(x1, x2, s1, s2, None, peers, rank, P, ob, tiling=t, trans_b=tb))
        assert L.last_launch().kernel == L.KERNEL_ALIGNED
    torch.cuda.synchronize()
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    want = x1[rank * rows:(rank + 1) * rows].float() @ (x2.T if tb else x2).float()   # (exact: |sums| < 2^24)
    assert torch.equal(got[0][1], want.to(torch.int32) + sum(peers))


# (rows per rank, N, K, P, rank, weights as [n,k], int32 peers): kept rows inside one 64-row tile, across two, at the end; two rows per wave column
@pytest.mark.parametrize("case", [(125, 516, 1376, 8, 5, True, False), (64, 260, 352, 8, 3, False, True), (18, 512, 416, 16, 0, True, False), (65, 1028, 100, 16, 8, False, False)])
@pytest.mark.parametrize("outbound", [False, True])
def test_reduce_scatter_peers_in_a_second_launch(case, outbound):
    """Ragged reduce-scatter launches of one round of tiles, with the workspace their query asks for: the kept rows' peers are added
    by a second launch.  The same sums in the same order as without a workspace: every output bit for bit, W8A8 also the oracle's."""
    _need_gpu()
    rows, N, K, P, rank, tb, ri = case
    M = rows * P
    rng = np.random.default_rng(rows + K)
    x1, x2 = rng.integers(-127, 128, (M, K), dtype=np.int8), rng.integers(-127, 128, (K, N), dtype=np.int8)
    s1, s2 = rng.uniform(0.005, 0.02, M).astype(np.float32), rng.uniform(0.001, 0.01, N).astype(np.float32)
    b = rng.integers(-1000, 1000, N, dtype=np.int32)
    peers = [rng.integers(-2 ** 24, 2 ** 24, (rows, N), dtype=np.int32) if ri else rng.standard_normal((rows, N)).astype(np.float32) for _ in range(P - 1)]
    acc, want = oracle.quant_matmul_reduce_scatter(x1, x2, s1, s2, b, rank * rows, rows, peers, oracle.BF16, reduce_int32=ri)
    t = ops.default_tiling(M, K, N, P, m0=0, n0=0, k0=0)
    d = L.make_desc(rank, P, [16] * (P - 1))
    tasks = L.load().catcoc_get_task_count(L.QUANT_MATMUL_REDUCE_SCATTER, C.byref(t), C.byref(d))
    size = L.load().catcoc_get_workspace_size(L.QUANT_MATMUL_REDUCE_SCATTER, L.INT8, C.byref(t), C.byref(d)) // 4
    flip = lambda w: np.ascontiguousarray(w.T) if tb else w
    dp = [dev(p) for p in peers]
    A, B = _rand16(rng, (M, K), oracle.FP16), _rand16(rng, (K, N), oracle.FP16, 0.02)
    bounds = sum_bound(A, B, oracle.FP16)
    for quant in (True, False) if not ri else (True,):
        need, f = ops.kslice_plan(L.QUANT_MATMUL_REDUCE_SCATTER if quant else L.MATMUL_REDUCE_SCATTER, torch.int8 if quant else torch.float16, M, K, N, rank, P, tiling=t)
        assert (need, f) == (65536 + rows * N * 4, 1) or f > 1
        got = []
        for ws in (torch.zeros(65536 + rows * N * 4, dtype=torch.uint8, device="cuda:0"), None):
            kw = {"outbound": torch.full((size,), 3, dtype=torch.int32 if ri else torch.float32, device="cuda:0")} if outbound else \
                 {"checksum": torch.full((tasks,), 77, dtype=torch.int64 if quant else torch.float64, device="cuda:0")}
            kw.update(tiling=t, trans_b=tb, workspace=ws, split_k=1)
            dump = torch.zeros((M, N), dtype=torch.int32 if quant else torch.float32, device="cuda:0")
            if quant:
                ca = torch.full((rows, N), -7, dtype=torch.int32, device="cuda:0")
                out = ops.quant_matmul_reduce_scatter(dev(x1), dev(flip(x2)), dev(s1), dev(s2), dev(b), dp, rank, P, reduce_int32=ri, c_accum=ca, acc_dump=dump, **kw)
                torch.cuda.synchronize()
                assert np.array_equal(host16(out), want) and np.array_equal(dump.cpu().numpy(), acc)
                assert np.array_equal(ca.cpu().numpy(), acc[rank * rows:(rank + 1) * rows] + (sum(peers) if ri else 0))
            else:
                out = ops.matmul_reduce_scatter(dev16(A, oracle.FP16), dev16(flip(B), oracle.FP16), dp, rank, P, acc_dump=dump, **kw)
                torch.cuda.synchronize()
                part, fwant = oracle.matmul_reduce(A, B, oracle.FP16, rank * rows, rows, peers, want_partial=True)
                _check_float(host16(out), fwant, part[rank * rows:(rank + 1) * rows] + sum(peers), oracle.FP16, K)
                assert (np.abs(dump.cpu().numpy() - part) <= bounds).all()
                for task, target, r0, c0, w0 in tasks_of(L.MATMUL_REDUCE_SCATTER, t, d):
                    at = np.s_[r0:min(r0 + (64 if rows <= 64 else 128), (target + 1) * rows), c0:min(c0 + 256, N)]
                    own = dump.cpu().numpy()[at]
                    if target != rank and outbound:
                        assert np.array_equal(kw["outbound"].cpu().numpy().reshape(-1, 256)[w0:w0 + own.shape[0], :own.shape[1]], own), task
                    elif target != rank:
                        assert abs(float(kw["checksum"][task]) - own.sum(dtype=np.float64)) <= own.size * 2.0 ** -51 * np.abs(own).sum(), task
            assert ws is None or (not ws[:65536].any() and bool(ws[65536:].any()))
            got.append([out, dump, kw.get("outbound", kw.get("checksum"))])
        for with_ws, without in zip(*got):
            assert torch.equal(with_ws, without)


# (kind, rows, N, K, P, kept rows or 0): launches whose flexible tiles would take k slices, or a second launch for the peers, that
# their query does not ask for: explicit kept rows off the 64/128 grid and in full tiles with a short k; aligned all-reduce with a k
# too short for the aligned kernel's slices; aligned reduce-scatter with stored tiles and a short k
@pytest.mark.parametrize("case", [("decode", 40, 260, 2052, 4, 40), ("decode", 130, 1100, 516, 2, 12), ("decode", 512, 1024, 768, 8, 512),
                                  ("allreduce", 512, 1024, 480, 2, 0), ("quant_rs", 1024, 4096, 256, 8, 0), ("float_rs", 1024, 4096, 128, 8, 0)])
@pytest.mark.parametrize("tb", [False, True])
def test_workspace_past_the_queried_bytes_is_not_touched(case, tb):
    """A launch uses no byte of a workspace past what its query says, also when that is none: the rest may be in use elsewhere."""
    _need_gpu()
    kind, M, N, K, P, kr = case
    g = torch.Generator(device="cuda:0").manual_seed(M + K)
    quant = kind in ("decode", "quant_rs")
    rows = kr or (M // P if kind.endswith("rs") else M)
    peers = [torch.randn((rows, N), device="cuda:0", generator=g) for _ in range(P - 1)]
    kw, rank = {}, P - 1
    if quant:
        a = torch.randint(-127, 128, (M, K), dtype=torch.int8, device="cuda:0", generator=g)
        b = torch.randint(-127, 128, (N, K) if tb else (K, N), dtype=torch.int8, device="cuda:0", generator=g)
        s1, s2 = (torch.empty(x, device="cuda:0").uniform_(0.001, 0.02, generator=g) for x in (M, N))
    else:
        a = torch.randn((M, K), device="cuda:0", generator=g).half()
        b = torch.randn((N, K) if tb else (K, N), device="cuda:0", generator=g).half()
    if kind == "decode":
        need = ops.splitk_plan(M, K, N, P, 0, kr)[0]
        run = lambda ws: ops.quant_matmul_splitk(a, b, s1, s2, None, peers, P, 0, kr, trans_b=tb, workspace=ws)
    else:
        comm, dt = {"allreduce": (L.MATMUL_ALLREDUCE, torch.float16), "quant_rs": (L.QUANT_MATMUL_REDUCE_SCATTER, torch.int8),
                    "float_rs": (L.MATMUL_REDUCE_SCATTER, torch.float16)}[kind]
        t = ops.default_tiling(M, K, N, P, m0=0, n0=0, k0=0)
        need = ops.kslice_plan(comm, dt, M, K, N, rank, P, tiling=t)[0]
        if kind != "allreduce":
            d = L.make_desc(rank, P, [16] * (P - 1))
            size = L.load().catcoc_get_workspace_size(comm, L.INT8 if quant else L.FP16, C.byref(t), C.byref(d)) // 4
            kw = {"outbound": torch.zeros(size, device="cuda:0")}
        if kind == "quant_rs":
            run = lambda ws: ops.quant_matmul_reduce_scatter(a, b, s1, s2, None, peers, rank, P, tiling=t, trans_b=tb, workspace=ws, **kw)
        elif kind == "float_rs":
            run = lambda ws: ops.matmul_reduce_scatter(a, b, peers, rank, P, tiling=t, trans_b=tb, workspace=ws, **kw)
        else:
            run = lambda ws: ops.matmul_allreduce(a, b, peers, rank, P, tiling=t, trans_b=tb, workspace=ws)
    end = max(need, 65536)
    got = []
    for extra in (0, 16 << 20):
        ws = torch.zeros(end + extra, dtype=torch.uint8, device="cuda:0")
        ws[65536:] = 0x55
        out = run(ws)
        torch.cuda.synchronize()
        assert bool((ws[end:] == 0x55).all()) and not ws[:65536].any()
        got.append(out.clone())
    assert torch.equal(got[0].view(torch.int16), got[1].view(torch.int16))


# (rows per rank, N, K, P, m0, ranks' tasks): several tasks in one tile (also with kept rows in its middle), tasks that cross from one
# wave's rows to the next, one task per tile, several tile rows per rank, k slices (a second launch) with all of these
@pytest.mark.parametrize("dtype", [oracle.FP16, oracle.BF16])
@pytest.mark.parametrize("case", [(11, 300, 200, 8, 0, 0), (1, 260, 132, 16, 0, 0), (63, 1028, 196, 4, 0, 0), (125, 516, 100, 8, 0, 0), (300, 516, 100, 4, 0, 0),
                                  (200, 300, 320, 2, 64, 0), (63, 512, 4112, 8, 0, 0), (11, 300, 200, 8, 0, 3), (150, 296, 4104, 4, 0, 0), (200, 300, 320, 2, 64, 2),
                                  (1, 260, 132, 16, 0, 2)])
def test_float_checksums_are_reproducible(case, dtype):
    """Checksums of float tiles: the sums of the dumped partials (64-bit sums in any order: 2^-52 of the magnitudes per addition),
    and the same bits in every launch.  Rows and columns differ in size by up to 2^20, so that these sums are not exact."""
    _need_gpu()
    rows, N, K, P, m0, slices = case
    M, rank = rows * P, P // 2
    g = torch.Generator(device="cuda:0").manual_seed(rows)
    size = lambda *shape: torch.exp2(-torch.randint(0, 11, shape, device="cuda:0", generator=g).float())
    A = (torch.randn((M, K), device="cuda:0", generator=g) * size(M, 1)).to(TORCH_DT[dtype])
    B = (torch.randn((K, N), device="cuda:0", generator=g) * size(1, N)).to(TORCH_DT[dtype])
    peers = [torch.randn((rows, N), device="cuda:0", generator=g) for _ in range(P - 1)]
    t = ops.default_tiling(M, K, N, P, m0=m0, n0=0, k0=0)
    d = L.make_desc(rank, P, [16] * (P - 1))
    tasks = L.load().catcoc_get_task_count(L.MATMUL_REDUCE_SCATTER, C.byref(t), C.byref(d))
    need, f = ops.kslice_plan(L.MATMUL_REDUCE_SCATTER, TORCH_DT[dtype], M, K, N, rank, P, tiling=t, split_k=slices)
    assert f == slices or (slices == 0 and (f > 1) == (K > 4000))
    ws = torch.zeros(max(need, 65536), dtype=torch.uint8, device="cuda:0")
    dump = torch.zeros((M, N), dtype=torch.float32, device="cuda:0")
    seen = []
    for _ in range(12):
        cs = torch.full((tasks,), 77.0, dtype=torch.float64, device="cuda:0")
        ops.matmul_reduce_scatter(A, B, peers, rank, P, tiling=t, checksum=cs, acc_dump=dump, workspace=ws, split_k=slices)
        torch.cuda.synchronize()
        seen.append(cs.cpu().numpy().view(np.int64))
    part = dump.cpu().numpy().astype(np.float64)
    step = m0 or (64 if rows <= 64 else 128)
    tr, row, col = C.c_uint32(), C.c_uint32(), C.c_uint32()
    for task in range(tasks):
        L.load().catcoc_task_tile(L.MATMUL_REDUCE_SCATTER, C.byref(t), C.byref(d), task, C.byref(tr), C.byref(row), C.byref(col), None)
        blk = part[row.value:min(row.value + step, (tr.value + 1) * rows), col.value:min(col.value + 256, N)]
        got = seen[0].view(np.float64)[task]
        if tr.value == rank:
            assert got == 77.0, task
        else:
            assert abs(got - blk.sum()) <= 2 * blk.size * 2.0 ** -52 * np.abs(blk).sum(), task
    assert all(np.array_equal(s, seen[0]) for s in seen[1:])


# (rows, N, K, P): ragged rows, ragged columns, whole k steps: the aligned kernels take these launches whole, their slices are flexible
@pytest.mark.parametrize("case", [(257, 512, 4096, 8), (300, 1032, 2048, 2)])
def test_ragged_launch_takes_the_slice_count_its_query_reports(case):
    _need_gpu()
    M, N, K, P = case
    g = torch.Generator(device="cuda:0").manual_seed(M)
    A, B = torch.randn((M, K), device="cuda:0", generator=g).bfloat16(), torch.randn((K, N), device="cuda:0", generator=g).bfloat16()
    peers = [torch.randn((M, N), device="cuda:0", generator=g) for _ in range(P - 1)]
    need, f = ops.kslice_plan(L.MATMUL_ALLREDUCE, torch.bfloat16, M, K, N, 0, P)
    outs = []
    for sk in (0, f):
        ws = torch.zeros(need, dtype=torch.uint8, device="cuda:0")
        out = ops.matmul_allreduce(A, B, peers, 0, P, workspace=ws, split_k=sk)
        torch.cuda.synchronize()
        assert f > 1 and bool(ws[65536:].any())
        outs.append(out)
    assert torch.equal(outs[0], outs[1])


# (rows per rank, N, K, P, rank, weights as [n,k], int32 peers, slices: 1 = peers in a second launch, swizzle)
@pytest.mark.parametrize("outbound", [False, True])
@pytest.mark.parametrize("case", [(125, 516, 1376, 8, 5, True, False, 1, (3, 0)), (125, 516, 1376, 8, 5, False, False, 3, (2, 1)), (40, 260, 516, 4, 1, False, True, 3, (1, 0)),
                                  (200, 1028, 260, 8, 2, True, True, 1, (2, 0)), (200, 772, 260, 8, 7, False, True, 4, (3, 1))])
def test_two_launches_with_a_window_of_the_peers_and_other_swizzles(case, outbound):
    """k slices and the peers' second launch: peers that are wider than n and start at a row of their own, other swizzles of the
    schedule, dumps and int32 sums."""
    _need_gpu()
    rows, N, K, P, rank, tb, ri, slices, swizzle = case
    M, off, step = rows * P, 5, 64 if rows <= 64 else 128
    rng = np.random.default_rng(rows + K + slices)
    x1, x2 = rng.integers(-127, 128, (M, K), dtype=np.int8), rng.integers(-127, 128, (K, N), dtype=np.int8)
    s1, s2 = rng.uniform(0.005, 0.02, M).astype(np.float32), rng.uniform(0.001, 0.01, N).astype(np.float32)
    b = rng.integers(-1000, 1000, N, dtype=np.int32)
    wide = [rng.integers(-2 ** 24, 2 ** 24, (rows + off + 2, N + 12), dtype=np.int32) if ri else rng.standard_normal((rows + off + 2, N + 12)).astype(np.float32)
            for _ in range(P - 1)]
    peers = [np.ascontiguousarray(p[off:off + rows, :N]) for p in wide]
    t = ops.default_tiling(M, K, N, P, m0=0, n0=0, k0=0)
    flip = lambda w: np.ascontiguousarray(w.T) if tb else w
    for quant in (True,) if ri else (True, False):
        comm = L.QUANT_MATMUL_REDUCE_SCATTER if quant else L.MATMUL_REDUCE_SCATTER
        d = L.make_desc(rank, P, [16] * (P - 1), swizzle=swizzle)
        tasks = list(tasks_of(comm, t, d))
        size = L.load().catcoc_get_workspace_size(comm, L.INT8 if quant else L.BF16, C.byref(t), C.byref(d)) // 4
        kw = {"outbound": torch.full((size,), 3, dtype=torch.int32 if ri else torch.float32, device="cuda:0")} if outbound else \
             {"checksum": torch.full((len(tasks),), 77, dtype=torch.int64 if quant else torch.float64, device="cuda:0")}
        ws = torch.zeros(65536 + (rows if slices == 1 else M * slices) * N * 4, dtype=torch.uint8, device="cuda:0")
        dump = torch.zeros((M, N), dtype=torch.int32 if quant else torch.float32, device="cuda:0")
        kw.update(tiling=t, trans_b=tb, workspace=ws, split_k=slices, swizzle=swizzle, peer_row_offset=off, acc_dump=dump)
        own = np.s_[rank * rows:(rank + 1) * rows]
        if quant:
            acc, want = oracle.quant_matmul_reduce_scatter(x1, x2, s1, s2, b, rank * rows, rows, peers, oracle.BF16, reduce_int32=ri)
            ca = torch.full((rows, N), -7, dtype=torch.int32, device="cuda:0")
            out = ops.quant_matmul_reduce_scatter(dev(x1), dev(flip(x2)), dev(s1), dev(s2), dev(b), [dev(p) for p in wide], rank, P, reduce_int32=ri, c_accum=ca, **kw)
            torch.cuda.synchronize()
            assert np.array_equal(host16(out), want) and np.array_equal(dump.cpu().numpy(), acc)
            assert np.array_equal(ca.cpu().numpy(), acc[own] + (sum(peers) if ri else 0))
            tiles = acc if ri or not outbound else oracle.dequant(acc, s2, s1)
        else:
            A, B = _rand16(rng, (M, K), oracle.BF16), _rand16(rng, (K, N), oracle.BF16, 0.02)
            part, want = oracle.matmul_reduce(A, B, oracle.BF16, rank * rows, rows, peers, want_partial=True)
            out = ops.matmul_reduce_scatter(dev16(A, oracle.BF16), dev16(flip(B), oracle.BF16), [dev(p) for p in wide], rank, P, **kw)
            torch.cuda.synchronize()
            _check_float(host16(out), want, part[own] + sum(peers), oracle.BF16, K)
            tiles = dump.cpu().numpy()
            assert (np.abs(tiles - part) <= sum_bound(A, B, oracle.BF16)).all()
        assert not ws[:65536].any() and bool(ws[65536:].any())
        for task, target, r0, c0, w0 in tasks:
            blk = tiles[r0:min(r0 + step, (target + 1) * rows), c0:min(c0 + 256, N)]
            if target == rank:
                assert outbound or int(kw["checksum"][task]) == 77
            elif outbound:
                got = kw["outbound"].cpu().numpy().reshape(-1, 256)[w0:w0 + blk.shape[0], :blk.shape[1]]
                assert np.array_equal(got.view(np.uint32), blk.view(np.uint32)), task
            elif quant:
                assert int(kw["checksum"][task]) == int(blk.astype(np.int64).sum()), task
            else:
                assert abs(float(kw["checksum"][task]) - blk.sum(dtype=np.float64)) <= blk.size * 2.0 ** -51 * np.abs(blk).sum(), task


# (M, N, K, P, kept rows [begin, +count), int32 peers): k and n off the 64/128 grid, no dump, sums of the rows that are not kept
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("case", [(130, 260, 1100, 2, 60, 11, False), (203, 416, 4100, 8, 0, 26, True), (203, 420, 416, 4, 190, 13, False), (40, 100, 132, 1, 3, 30, False)])
def test_quant_kept_rows_off_the_grid_without_a_dump(case, tb):
    _need_gpu()
    M, N, K, P, kb, kr, ri = case
    rng = np.random.default_rng(M + K)
    x1, x2 = rng.integers(-127, 128, (M, K), dtype=np.int8), rng.integers(-127, 128, (K, N), dtype=np.int8)
    s1, s2 = rng.uniform(0.005, 0.02, M).astype(np.float32), rng.uniform(0.001, 0.01, N).astype(np.float32)
    b = rng.integers(-1000, 1000, N, dtype=np.int32)
    peers = [rng.integers(-2 ** 24, 2 ** 24, (kr, N), dtype=np.int32) if ri else rng.standard_normal((kr, N)).astype(np.float32) for _ in range(P - 1)]
    acc, want = oracle.quant_matmul_reduce_scatter(x1, x2, s1, s2, b, kb, kr, peers, oracle.BF16, reduce_int32=ri)
    cs = torch.full((-(-M // 128) * -(-N // 128),), -7, dtype=torch.int64, device="cuda:0")
    ca = torch.full((kr, N), -7, dtype=torch.int32, device="cuda:0")
    out = ops.quant_matmul_splitk(dev(x1), dev(np.ascontiguousarray(x2.T) if tb else x2), dev(s1), dev(s2), dev(b), [dev(p) for p in peers], P, kb, kr,
                                  checksum=cs, c_accum=ca, trans_b=tb, reduce_int32=ri)
    torch.cuda.synchronize()
    assert np.array_equal(host16(out), want) and np.array_equal(ca.cpu().numpy(), acc[kb:kb + kr] + (sum(peers) if ri else 0))
    others = acc.astype(np.int64)
    others[kb:kb + kr] = 0
    assert np.array_equal(cs.cpu().numpy(), [others[r:r + 128, c:c + 128].sum() for r in range(0, M, 128) for c in range(0, N, 128)])


# (rows per rank, N, K, P, rank, weights as [n,k])
@pytest.mark.parametrize("case", [(128, 640, 448, 8, 3, False), (256, 1440, 192, 4, 0, True), (72, 288, 100, 2, 1, False), (128, 512, 1024, 8, 7, True)])
@pytest.mark.parametrize("dtype", [oracle.FP16, oracle.BF16])
def test_pipelined_float_one_round(case, dtype):
    """One-round calls of the 16-bit pipelined operator on ragged columns, ragged rows and few aligned tiles: the reduced block as
    the oracle replays it from the dumped partials, the other ranks' tiles as they were dumped."""
    _need_gpu()
    rows, N, K, P, rank, tb = case
    M = rows * P
    rng = np.random.default_rng(rows + N)
    A, B = _rand16(rng, (M, K), dtype), _rand16(rng, (K, N), dtype, 0.05)
    peers = [_rand16(rng, (rows, N), dtype) for _ in range(P - 1)]
    t = ops.default_tiling(M, K, N, P, m0=128, n0=256, k0=0, commInterval=1)
    d = L.make_desc(rank, P, [16] * (P - 1))
    assert ops.pipelined_round_count(L.MATMUL_REDUCE_SCATTER, t, rank, P) == 1
    ob = torch.full((L.load().catcoc_get_workspace_size(L.MATMUL_REDUCE_SCATTER, dtype, C.byref(t), C.byref(d)) // 4,), -9.0, device="cuda:0")
    dump = torch.zeros((M, N), dtype=torch.float32, device="cuda:0")
    out = ops.pipelined_matmul_reduce_scatter(dev16(A, dtype), dev16(np.ascontiguousarray(B.T) if tb else B, dtype), [dev16(p, dtype) for p in peers], rank, P, ob,
                                              tiling=t, trans_b=tb, acc_dump=dump)
    torch.cuda.synchronize()
    part = dump.cpu().numpy()
    assert (np.abs(part - oracle.gemm_half_f32(A, B, dtype)) <= sum_bound(A, B, dtype)).all()
    assert np.array_equal(host16(out), oracle.pipelined_reduce_half(part[rank * rows:(rank + 1) * rows], peers, dtype, M, P, rank, 128, 256, 256, 1, 64, 256, 1))
    for task, target, r0, c0, w0 in tasks_of(L.MATMUL_REDUCE_SCATTER, t, d):
        if target != rank:
            blk = part[r0:min(r0 + 128, (target + 1) * rows), c0:min(c0 + 256, N)]
            assert np.array_equal(ob.cpu().numpy().reshape(-1, 256)[w0:w0 + blk.shape[0], :blk.shape[1]], blk), task


def test_launches_of_several_kernels_replay_from_a_hip_graph():
    """Flexible launches of two and three kernels (k slices, the peers' second launch, the sums of float tasks): every replay, with
    eager work in between, equals the eager result."""
    _need_gpu()
    g = torch.Generator(device="cuda:0").manual_seed(3)
    rand = lambda *shape: torch.randn(shape, device="cuda:0", generator=g)
    byte = lambda *shape: torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda:0", generator=g)
    scale = lambda n: torch.empty(n, device="cuda:0").uniform_(0.001, 0.02, generator=g)
    state = []

    def call(fn, outputs, need):
        ws = torch.zeros(max(need, 65536), dtype=torch.uint8, device="cuda:0")
        state.append((lambda: fn(ws), outputs, ws))
    # float reduce-scatter with checksums in slices, the same with stored tiles
    P, rows, N, K = 8, 63, 516, 4112
    A, B, peers = rand(P * rows, K).bfloat16(), rand(K, N).bfloat16(), [rand(rows, N) for _ in range(P - 1)]
    t = ops.default_tiling(P * rows, K, N, P, m0=0, n0=0, k0=0)
    need, f = ops.kslice_plan(L.MATMUL_REDUCE_SCATTER, torch.bfloat16, P * rows, K, N, 1, P, tiling=t)
    assert f > 2
    cs, out = torch.zeros(P * 3, dtype=torch.float64, device="cuda:0"), torch.zeros((rows, N), dtype=torch.bfloat16, device="cuda:0")
    call(lambda ws: ops.matmul_reduce_scatter(A, B, peers, 1, P, tiling=t, checksum=cs, out=out, workspace=ws), [out, cs], need)
    # W8A8 reduce-scatter, the peers in a second launch
    x1, x2, s1, s2 = byte(1000, 352), byte(352, 516), scale(1000), scale(516)
    qpeers = [rand(125, 516) for _ in range(7)]
    need, f = ops.kslice_plan(L.QUANT_MATMUL_REDUCE_SCATTER, torch.int8, 1000, 352, 516, 5, 8)
    qout, qcs = torch.zeros((125, 516), dtype=torch.bfloat16, device="cuda:0"), torch.zeros(24, dtype=torch.int64, device="cuda:0")
    assert f == 1 and need > 65536 or f > 1
    call(lambda ws: ops.quant_matmul_reduce_scatter(x1, x2, s1, s2, None, qpeers, 5, 8, checksum=qcs, out=qout, workspace=ws), [qout, qcs], need)
    # all-reduce in slices, W8A8 decode in slices with sums of the other rows
    need, f = ops.kslice_plan(L.MATMUL_ALLREDUCE, torch.float16, 33, 4096, 512, 0, 2)
    a, b, ap, ao = rand(33, 4096).half(), rand(4096, 512).half(), [rand(33, 512)], torch.zeros((33, 512), dtype=torch.float16, device="cuda:0")
    assert f > 1
    call(lambda ws: ops.matmul_allreduce(a, b, ap, 0, 2, out=ao, workspace=ws), [ao], need)
    d1, d2, e1, e2 = byte(130, 1024), byte(1024, 640), scale(130), scale(640)
    dp, do, dcs = [rand(12, 640)], torch.zeros((12, 640), dtype=torch.bfloat16, device="cuda:0"), torch.zeros(10, dtype=torch.int64, device="cuda:0")
    need = ops.splitk_plan(130, 1024, 640, 2, 60, 12)[0]
    call(lambda ws: ops.quant_matmul_splitk(d1, d2, e1, e2, None, dp, 2, 60, 12, checksum=dcs, out=do, workspace=ws), [do, dcs], need)

    for fn, _, _ in state:
        fn()
    torch.cuda.synchronize()
    want = [[o.clone() for o in outputs] for _, outputs, _ in state]
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(side):
        for fn, _, _ in state:
            fn()
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=side):
            for fn, _, _ in state:
                fn()
    for replay in range(3):
        for fn, outputs, ws in state:
            for o in outputs:
                o.fill_(replay + 1)
            ws[65536:] = 0x3c   # (what an earlier launch left there does not matter)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for (fn, outputs, ws), w in zip(state, want):
            for o, x in zip(outputs, w):
                same = (o == x) | (o == replay + 1) if o.dim() == 1 else o == x   # (sums of the kept rank's tasks are not written)
                assert bool(same.all()) and not ws[:65536].any()
        for fn, _, _ in state:   # eager work between the replays
            fn()
        torch.cuda.synchronize()


@pytest.mark.parametrize("slices", [0, 3])
@pytest.mark.parametrize("tb", [False, True])
def test_values_that_are_not_finite_stay_in_their_rows_and_columns(slices, tb):
    """Rows and columns past the edge of a tile repeat the last one and rows of B are read past their end: an infinity or NaN there
    reaches no other row or column, nor do those of the k remainder or of peers."""
    _need_gpu()
    M, N, K, P = 65, 260, 1028, 3
    rng = np.random.default_rng(9)
    A, B = _rand16(rng, (M, K), oracle.FP16, 1.0), _rand16(rng, (K, N), oracle.FP16, 0.02)
    inf, nan = 0x7c00, 0x7e00
    A[64, 3], A[0, K - 1], B[5, 259], B[K - 1, 7] = inf, nan, inf, nan
    peers = [rng.standard_normal((M, N)).astype(np.float32) for _ in range(P - 1)]
    peers[0][63, 100], peers[1][10, 258] = np.inf, np.nan
    ws = torch.zeros(65536 + 3 * M * N * 4, dtype=torch.uint8, device="cuda:0") if slices else None
    out = ops.matmul_allreduce(dev16(A, oracle.FP16), dev16(np.ascontiguousarray(B.T) if tb else B, oracle.FP16), [dev(p) for p in peers], 0, P, trans_b=tb,
                               workspace=ws, split_k=slices)
    torch.cuda.synchronize()
    with np.errstate(invalid="ignore"):
        want = oracle.half_to_f32(A, oracle.FP16).astype(np.float64) @ oracle.half_to_f32(B, oracle.FP16).astype(np.float64) + peers[0] + peers[1]
    got = oracle.half_to_f32(host16(out), oracle.FP16)
    finite = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isfinite(got), finite) and np.array_equal(np.sign(got[np.isinf(want)]), np.sign(want[np.isinf(want)]))
    assert (np.abs(got[finite] - want[finite]) <= 2.0 ** -10 * np.abs(want[finite]) + 4e-3).all()   # (one rounding to fp16, fp32 sums as in sum_bound)
    assert (~finite).sum() == 2 * N + 2 * (M - 2) + 2


# (M, N, K, P, kept rows, checksums): explicit kept rows on both sides of every line between the streaming kernels and flexible tiles
@pytest.mark.parametrize("case", [(32, 4096, 4096, 2, 32, False), (32, 6272, 4096, 2, 8, True), (33, 256, 256, 2, 33, False), (33, 256, 256, 3, 33, False),
                                  (48, 128, 448, 8, 48, False), (64, 384, 256, 1, 8, False), (64, 384, 256, 1, 8, True), (64, 384, 320, 2, 8, True),
                                  (64, 384, 320, 3, 8, True), (128, 256, 320, 8, 16, False), (128, 256, 256, 8, 64, False), (128, 256, 448, 8, 63, False),
                                  (256, 256, 448, 8, 128, False), (256, 256, 448, 8, 96, False), (256, 256, 448, 2, 128, True), (384, 1536, 4096, 1, 384, False),
                                  (512, 8448, 128, 2, 256, False)])
@pytest.mark.parametrize("tb", [False, True])
def test_decode_on_both_sides_of_the_choice_of_kernels(case, tb):
    _need_gpu()
    M, N, K, P, kr, sums = case
    rng = np.random.default_rng(M + K)
    x1, x2 = rng.integers(-127, 128, (M, K), dtype=np.int8), rng.integers(-127, 128, (K, N), dtype=np.int8)
    s1, s2 = rng.uniform(0.005, 0.02, M).astype(np.float32), rng.uniform(0.001, 0.01, N).astype(np.float32)
    peers = [rng.standard_normal((kr, N)).astype(np.float32) for _ in range(P - 1)]
    acc, want = oracle.quant_matmul_reduce_scatter(x1, x2, s1, s2, None, 0, kr, peers, oracle.BF16)
    need, _, tiles = ops.splitk_plan(M, K, N, P, 0, kr)
    ws = torch.zeros(max(need, 65536), dtype=torch.uint8, device="cuda:0")
    cs = torch.full((tiles,), -7, dtype=torch.int64, device="cuda:0") if sums else None
    ca = torch.full((kr, N), -7, dtype=torch.int32, device="cuda:0")
    out = ops.quant_matmul_splitk(dev(x1), dev(np.ascontiguousarray(x2.T) if tb else x2), dev(s1), dev(s2), None, [dev(p) for p in peers], P, 0, kr, workspace=ws,
                                  checksum=cs, c_accum=ca, trans_b=tb)
    torch.cuda.synchronize()
    assert np.array_equal(host16(out), want) and np.array_equal(ca.cpu().numpy(), acc[:kr]) and not ws[:65536].any()
    if sums:
        acc[:kr] = 0
        assert np.array_equal(cs.cpu().numpy(), [acc[r:r + 128, c:c + 128].astype(np.int64).sum() for r in range(0, M, 128) for c in range(0, N, 128)])


# (M, N, K, P): stored tiles without a workspace, kept tiles that the aligned kernel splits, k and tile counts around the lines
@pytest.mark.parametrize("case", [(512, 4096, 1024, 4), (512, 4096, 1088, 4), (768, 4096, 2048, 2), (768, 4096, 2112, 2), (1024, 2048, 1024, 8)])
@pytest.mark.parametrize("tb", [False, True])
def test_stored_tiles_on_both_sides_of_the_choice_of_kernels(case, tb):
    M, N, K, P = case
    t = ops.default_tiling(M, K, N, P, m0=0, n0=0, k0=0)
    r = quant_case(np.random.default_rng(K), M, N, K, P, P - 1, trans_b=tb, tiling=t, outbound=True)
    assert r["exact"] == r["total"]
    d = L.make_desc(P - 1, P, [16] * (P - 1))
    deq, ob = oracle.dequant(r["acc"], r["s2"], r["s1"]), r["outbound"].cpu().numpy().reshape(-1, 256)
    for task, target, r0, c0, w0 in tasks_of(L.QUANT_MATMUL_REDUCE_SCATTER, t, d):
        if target != P - 1:
            assert np.array_equal(ob[w0:w0 + 128].view(np.uint32), deq[r0:r0 + 128, c0:c0 + 256].view(np.uint32)), task


@pytest.fixture
def flexible(monkeypatch):
    """Ragged calls of the operators in the schedule's order: on flexible tiles, where small ones would else take some.  Every launch is seen to run there."""
    def ordered(op):
        def call(*a, **kw):
            out = op(*a, **dict(kw, linear_order=True))
            assert L.last_launch().kernel == L.KERNEL_FLEXIBLE
            return out
        return call
    for name in ("matmul_allreduce", "allgather_matmul", "quant_matmul_reduce_scatter"):
        monkeypatch.setattr(ops, name, ordered(getattr(ops, name)))


@pytest.mark.parametrize("dtype", [oracle.FP16, oracle.BF16])
@pytest.mark.parametrize("case", [("allreduce", 1, 256, 128, 8, True), ("allgather", 3, 264, 516, 8, True), ("allgather", 65, 768, 1026, 4, False)])
def test_float_any_rows_any_k_on_flexible_tiles(dtype, case, flexible):
    test_float_any_rows_any_k(dtype, case)


@pytest.mark.parametrize("case", [(125, 512, 1376, 8, 5, True, False, 0, 1), (8, 256, 64, 8, 0, False, True, 0, 1), (65, 772, 260, 8, 7, True, True, 0, 1), (300, 516, 100, 4, 3, True, False, 0, 1)])
def test_quant_rs_any_rows_any_k_on_flexible_tiles(case, flexible):
    test_quant_rs_any_rows_any_k(case, True)


def test_values_that_are_not_finite_on_flexible_tiles(flexible):
    test_values_that_are_not_finite_stay_in_their_rows_and_columns(0, True)
