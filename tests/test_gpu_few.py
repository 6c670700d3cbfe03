"""GPU parity of the one-launch kernels for small tiles (csrc/gemm_few.h, csrc/gemm_mid.h) and for mixed ones (csrc/gemm_mixed.h) at the edges of their tiles and of k: W8A8 outputs,
workspace tiles and dumps bit for bit, float sums within the bound of two orders of the same additions."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle
from mm_rs_with_catlass_amd import lib as L
from mm_rs_with_catlass_amd import ops
from test_gpu_flex import sum_bound, tasks_of
from test_gpu_parity import _need_gpu, _rand16, dev, dev16, host16

pytestmark = pytest.mark.gpu


def ran():
    """The tiles that the last launch ran, as the cases name them: those of another kernel than this file's with its name, k slices behind a stroke,
    256x256 ones beside 128x128 ones."""
    i = L.last_launch()
    kernel = {L.KERNEL_SMALL: "", L.KERNEL_FLEXIBLE: "flexible ", L.KERNEL_ALIGNED: "aligned ", L.KERNEL_STREAMING: "streaming "}[i.kernel]
    assert (i.largeTiles != 0) == (i.kernel == L.KERNEL_SMALL and i.tileRows == 256)
    return "%s%dx%d%s%s" % (kernel, i.tileRows, i.tileCols, "/%d" % i.kSlices if i.kSlices > 1 else "", " dealt" if i.dealt else "")


# (rows, N, K, P, weights as [n,k]): one row; a tile less, full, one more; columns that end inside a tile and a 16-byte piece of the
# output; k of one piece, less than a chunk, 4, 8 and 12 bytes into a piece (the first of a chunk, a later one), fewer chunks than waves; tiles of 32x64 and 64x64
@pytest.mark.parametrize("dtype", [oracle.FP16, oracle.BF16])
@pytest.mark.parametrize("case", [(1, 4, 8, 2, True, "32x32"), (1, 36, 514, 8, True, "32x32"), (31, 32, 64, 3, False, "32x32"), (32, 264, 66, 16, False, "32x32"),
                                  (33, 100, 324, 8, True, "32x32"), (64, 4096, 128, 2, True, "32x32"), (65, 1032, 1030, 4, False, "32x32"),
                                  (129, 72, 2052, 11, False, "32x32"), (200, 3996, 192, 1, True, "64x64"), (407, 1256, 160, 2, False, "64x64"),
                                  (290, 1064, 1034, 3, False, "32x64"), (203, 1376, 84, 3, True, "32x64"), (370, 1688, 124, 2, True, "64x64")])
def test_float_allreduce(case, dtype):
    _need_gpu()
    M, N, K, P, tb, tiles = case
    rng = np.random.default_rng(M + K)
    A, B = _rand16(rng, (M, K), dtype), _rand16(rng, (K, N), dtype, 0.05)
    peers = [rng.standard_normal((M + 3, N + 4)).astype(np.float32) for _ in range(P - 1)]
    dump = torch.full((M, N), 7.0, dtype=torch.float32, device="cuda:0")
    out = ops.matmul_allreduce(dev16(A, dtype), dev16(np.ascontiguousarray(B.T) if tb else B, dtype), [dev(p) for p in peers], 0, P, trans_b=tb,
                               peer_row_offset=3, acc_dump=dump)
    assert ran() == tiles
    torch.cuda.synchronize()
    got, want = dump.cpu().numpy(), oracle.half_to_f32(A, dtype).astype(np.float64) @ oracle.half_to_f32(B, dtype).astype(np.float64)
    assert (np.abs(got - want) <= sum_bound(A, B, dtype)).all()
    for p in peers:   # from the kernel's own sums on every step has one right answer
        got = got + p[3:, :N]
    assert np.array_equal(host16(out), oracle.f32_to_half(got, dtype))


@pytest.mark.parametrize("case", [(1, 260, 130, 8, True, "32x32"), (7, 64, 256, 5, False, "32x32"), (33, 136, 1028, 2, True, "32x32"), (40, 520, 98, 3, False, "32x32"),
                                  (257, 280, 102, 4, False, "32x64"), (112, 1328, 108, 2, True, "32x64"), (92, 1928, 146, 3, False, "64x64"),
                                  (275, 488, 96, 4, True, "64x64"), (256, 1644, 400, 3, True, "64x128"), (271, 1944, 832, 2, False, "64x128")])
def test_float_allgather_tiles_across_shards(case):
    _need_gpu()
    m, N, K, P, tb, tiles = case
    rng = np.random.default_rng(m + K)
    B = _rand16(rng, (K, N), oracle.BF16, 0.05)
    shards = [_rand16(rng, (m, K), oracle.BF16) for _ in range(P)]
    rank = P // 2
    ds = [dev16(s, oracle.BF16) for s in shards]
    dump = torch.full((m * P, N), 7.0, dtype=torch.float32, device="cuda:0")
    out = ops.allgather_matmul(ds[rank], ds[:rank] + ds[rank + 1:], dev16(np.ascontiguousarray(B.T) if tb else B, oracle.BF16), rank, P, trans_b=tb, acc_dump=dump)
    assert ran() == tiles
    torch.cuda.synchronize()
    A = np.concatenate(shards)
    want = oracle.half_to_f32(A, oracle.BF16).astype(np.float64) @ oracle.half_to_f32(B, oracle.BF16).astype(np.float64)
    assert (np.abs(dump.cpu().numpy() - want) <= sum_bound(A, B, oracle.BF16)).all()
    assert np.array_equal(host16(out), oracle.f32_to_half(dump.cpu().numpy(), oracle.BF16))


# (rows, N, K, P, first kept row, kept rows, weights as [n,k], int32 peers)
@pytest.mark.parametrize("case", [(1, 128, 128, 8, 0, 1, True, False, "32x32"), (17, 384, 1344, 16, 3, 9, True, True, "32x32"),
                                  (32, 36, 20, 2, 31, 1, True, False, "32x32"), (33, 260, 1236, 4, 30, 3, False, True, "flexible 64x256"),
                                  (70, 48, 260, 8, 0, 70, False, False, "32x32"), (203, 1792, 1776, 8, 64, 100, False, False, "32x64"),
                                  (336, 1696, 140, 3, 0, 336, False, True, "64x64"), (286, 1964, 124, 5, 0, 286, True, False, "64x64"),
                                  (645, 2608, 1344, 2, 0, 645, False, False, "64x128"), (514, 2224, 2092, 2, 0, 514, True, False, "64x128"),
                                  (387, 1424, 80, 4, 0, 387, False, False, "64x64")])
def test_quant_kept_rows(case):
    _need_gpu()
    M, N, K, P, kb, kr, tb, ri, tiles = case
    rng = np.random.default_rng(M + N)
    x1, x2 = rng.integers(-127, 128, (M, K), dtype=np.int8), rng.integers(-127, 128, (K, N), dtype=np.int8)
    s1, s2 = rng.uniform(0.005, 0.02, M).astype(np.float32), rng.uniform(0.001, 0.01, N).astype(np.float32)
    b = rng.integers(-1000, 1000, N, dtype=np.int32)
    peers = [rng.integers(-2 ** 24, 2 ** 24, (kr, N), dtype=np.int32) if ri else rng.standard_normal((kr, N)).astype(np.float32) for _ in range(P - 1)]
    acc, want = oracle.quant_matmul_reduce_scatter(x1, x2, s1, s2, b, kb, kr, peers, oracle.BF16, reduce_int32=ri)
    dump = torch.full((M, N), -7, dtype=torch.int32, device="cuda:0")
    need = ops.splitk_plan(M, K, N, P, kb, kr)[0]
    ws = torch.zeros(max(need, 65536), dtype=torch.uint8, device="cuda:0")
    out = ops.quant_matmul_splitk(dev(x1), dev(np.ascontiguousarray(x2.T) if tb else x2), dev(s1), dev(s2), dev(b), [dev(p) for p in peers], P, kb, kr,
                                  workspace=ws, acc_dump=dump, trans_b=tb, reduce_int32=ri)
    assert ran() == tiles
    torch.cuda.synchronize()
    assert np.array_equal(host16(out), want) and np.array_equal(dump.cpu().numpy(), acc) and not ws[:65536].any()

# The peers are asked for at once where a wave's chunks of 128 bytes of k fill its ring at most (20 chunks of 32x32 tiles, 12 of 32x64, 8 of 64x64),
# behind the first copies else; seven (64x64) or eight of them are held in registers.
@pytest.mark.parametrize("case", [(33, 1344, 2560, 8, 0, 33, True, False, "32x32"), (33, 1344, 2564, 9, 5, 20, True, False, "32x32"), (33, 1344, 2560, 10, 0, 33, False, True, "32x32"),
                                  (250, 1376, 1536, 8, 0, 250, True, False, "32x64"), (250, 1376, 1540, 9, 40, 100, True, True, "32x64"),
                                  (250, 1376, 1536, 10, 0, 250, False, False, "32x64"),
                                  (330, 1696, 1024, 8, 0, 330, True, False, "64x64"), (330, 1696, 1028, 9, 60, 70, True, False, "64x64"),
                                  (330, 1696, 1020, 9, 0, 330, False, True, "64x64")])
def test_quant_peers_at_once_or_in_turn(case):
    test_quant_kept_rows(case)



# (rows per rank, N, K, P, rank, weights as [n,k], int32 peers): kept rows inside a tile and across two, other ranks' rows beside them
@pytest.mark.parametrize("case", [(5, 260, 132, 8, 3, True, False, "32x32", "32x32"), (20, 512, 416, 4, 0, False, True, "32x32", "32x32"),
                                  (33, 300, 1000, 16, 15, True, False, "32x32", "32x32"), (61, 128, 272, 2, 1, False, False, "32x32", "32x32")])
def test_reduce_scatter_stored_tiles(case):
    _need_gpu()
    rows, N, K, P, rank, tb, ri, *kinds = case
    M = rows * P
    rng = np.random.default_rng(M + N)
    flip = lambda w: np.ascontiguousarray(w.T) if tb else w
    x1, x2 = rng.integers(-127, 128, (M, K), dtype=np.int8), rng.integers(-127, 128, (K, N), dtype=np.int8)
    s1, s2 = rng.uniform(0.005, 0.02, M).astype(np.float32), rng.uniform(0.001, 0.01, N).astype(np.float32)
    b = rng.integers(-1000, 1000, N, dtype=np.int32)
    peers = [rng.integers(-2 ** 24, 2 ** 24, (rows, N), dtype=np.int32) if ri else rng.standard_normal((rows, N)).astype(np.float32) for _ in range(P - 1)]
    acc, want = oracle.quant_matmul_reduce_scatter(x1, x2, s1, s2, b, rank * rows, rows, peers, oracle.BF16, reduce_int32=ri)
    A, B = _rand16(rng, (M, K), oracle.FP16), _rand16(rng, (K, N), oracle.FP16, 0.05)
    t = ops.default_tiling(M, K, N, P, m0=0, n0=0, k0=0)
    d = L.make_desc(rank, P, [16] * (P - 1))
    for quant in (True,) if ri else (True, False):
        comm = L.QUANT_MATMUL_REDUCE_SCATTER if quant else L.MATMUL_REDUCE_SCATTER
        size = L.load().catcoc_get_workspace_size(comm, L.INT8 if quant else L.FP16, C.byref(t), C.byref(d)) // 4
        ob = torch.full((size,), 3, dtype=torch.int32 if ri else torch.float32, device="cuda:0")
        if quant:
            sums = torch.full((rows, N), -7, dtype=torch.int32, device="cuda:0")
            out = ops.quant_matmul_reduce_scatter(dev(x1), dev(flip(x2)), dev(s1), dev(s2), dev(b), [dev(p) for p in peers], rank, P, tiling=t, trans_b=tb,
                                                  reduce_int32=ri, outbound=ob, c_accum=sums)
            full = acc if ri else oracle.dequant(acc, s2, s1)
            kept = acc[rank * rows:(rank + 1) * rows] + (sum(peers) if ri else 0)
            assert np.array_equal(host16(out), want) and np.array_equal(sums.cpu().numpy(), kept)
        else:
            dump = torch.zeros((M, N), dtype=torch.float32, device="cuda:0")
            out = ops.matmul_reduce_scatter(dev16(A, oracle.FP16), dev16(flip(B), oracle.FP16), [dev(p) for p in peers], rank, P, tiling=t, trans_b=tb,
                                            outbound=ob, acc_dump=dump)
            full = dump.cpu().numpy()
            exact = oracle.half_to_f32(A, oracle.FP16).astype(np.float64) @ oracle.half_to_f32(B, oracle.FP16).astype(np.float64)
            assert (np.abs(full - exact) <= sum_bound(A, B, oracle.FP16)).all()
            got = full[rank * rows:(rank + 1) * rows]
            for p in peers:
                got = got + p
            assert np.array_equal(host16(out), oracle.f32_to_half(got, oracle.FP16))
        assert ran() == kinds[0 if quant else 1]
        step = 64 if rows <= 64 else 128
        tiles = ob.cpu().numpy().reshape(-1, 256)
        for task, r, row, col, ws in tasks_of(comm, t, d):
            if r != rank:
                r1, c1 = min(row + step, (r + 1) * rows), min(col + 256, N)
                assert np.array_equal(tiles[ws:ws + r1 - row, :c1 - col].view(np.uint32), full[row:r1, col:c1].view(np.uint32)), task


@pytest.mark.parametrize("case", [(35, 72, 586, 4, True, "32x32"), (35, 72, 586, 4, False, "32x32"), (3, 40, 1024, 2, True, "32x32")])
def test_values_that_are_not_finite_stay_in_their_row_and_column(case):
    """Infinities in the last element of k: the pieces past the end of k hold them too and must not reach a sum."""
    _need_gpu()
    M, N, K, P, tb, tiles = case
    rng = np.random.default_rng(K)
    A, B = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((K, N)).astype(np.float32)
    A[M // 2, K - 1], B[K - 1, N // 3], B[K - 17, 1] = -np.inf, np.inf, np.nan
    ab, bb = oracle.f32_to_half(A, oracle.BF16), oracle.f32_to_half(B, oracle.BF16)
    peers = [rng.standard_normal((M, N)).astype(np.float32) for _ in range(P - 1)]
    out = ops.matmul_allreduce(dev16(ab, oracle.BF16), dev16(np.ascontiguousarray(bb.T) if tb else bb, oracle.BF16), [dev(p) for p in peers], 0, P, trans_b=tb)
    assert ran() == tiles
    torch.cuda.synchronize()
    got = oracle.half_to_f32(host16(out), oracle.BF16)
    with np.errstate(all="ignore"):
        want = oracle.half_to_f32(ab, oracle.BF16).astype(np.float64) @ oracle.half_to_f32(bb, oracle.BF16).astype(np.float64) + sum(peers)
    fin = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), fin) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    assert (np.abs(got[fin] - want[fin]) <= 2.0 ** -8 * np.abs(want[fin]) + 1e-2).all()   # (half a last place of 8 bits, and the sums' own bound)


# (rows, N, K, P, first kept row, kept rows, weights as [n,k], tiles): checksums of tiles smaller than a block and as large, with a dump; rows
# and columns one past a tile, k of one chunk and less, of a few bytes more than whole chunks, more chunks than stages
@pytest.mark.parametrize("case", [(40, 128, 100, 2, 3, 10, True, "32x32"), (64, 132, 132, 8, 0, 8, True, "32x32"), (65, 260, 1236, 4, 60, 5, False, "flexible 128x256"),
                                  (128, 112, 776, 3, 88, 40, False, "32x32"), (129, 516, 648, 8, 128, 1, True, "32x32"), (300, 240, 2440, 6, 100, 150, False, "32x32"),
                                  (18, 48, 36, 1, 2, 4, True, "32x32"), (454, 2416, 96, 16, 101, 1, False, "64x128"), (560, 2132, 112, 8, 37, 330, True, "64x128"),
                                  (700, 4608, 1296, 2, 130, 300, False, "128x128"), (650, 4612, 1292, 3, 600, 50, True, "128x128")])
def test_quant_kept_rows_with_checksums(case):
    _need_gpu()
    M, N, K, P, kb, kr, tb, tiles = case
    rng = np.random.default_rng(M + N)
    x1, x2 = rng.integers(-127, 128, (M, K), dtype=np.int8), rng.integers(-127, 128, (K, N), dtype=np.int8)
    s1, s2 = rng.uniform(0.005, 0.02, M).astype(np.float32), rng.uniform(0.001, 0.01, N).astype(np.float32)
    b = rng.integers(-1000, 1000, N, dtype=np.int32)
    peers = [rng.standard_normal((kr, N)).astype(np.float32) for _ in range(P - 1)]
    acc, want = oracle.quant_matmul_reduce_scatter(x1, x2, s1, s2, b, kb, kr, peers, oracle.BF16)
    others = acc.astype(np.int64)
    others[kb:kb + kr] = 0
    sums = np.array([others[r:r + 128, c:c + 128].sum() for r in range(0, M, 128) for c in range(0, N, 128)])
    cs = torch.full((sums.size,), -7, dtype=torch.int64, device="cuda:0")
    dump = torch.full((M, N), -7, dtype=torch.int32, device="cuda:0")
    out = ops.quant_matmul_splitk(dev(x1), dev(np.ascontiguousarray(x2.T) if tb else x2), dev(s1), dev(s2), dev(b), [dev(p) for p in peers], P, kb, kr,
                                  workspace=torch.zeros(1 << 20, dtype=torch.uint8, device="cuda:0"), checksum=cs, acc_dump=dump, trans_b=tb)
    assert ran() == tiles
    torch.cuda.synchronize()
    assert np.array_equal(host16(out), want) and np.array_equal(dump.cpu().numpy(), acc) and np.array_equal(cs.cpu().numpy(), sums)


def marked(rows, N, dtype):
    """An output that says which of its elements a launch left alone."""
    return torch.full((rows, N), 12345.0, dtype=dtype, device="cuda:0")


def one_round(comm, M, K, N, P, rank):
    """Tiling and descriptor of a call whose tiles all have a place of their own in the symmetric workspace."""
    t, d = ops.default_tiling(M, K, N, P, m0=0, n0=0, k0=0), L.make_desc(rank, P, [16] * (P - 1))
    t.commInterval = max(1, -(-L.load().catcoc_get_task_count(comm, C.byref(t), C.byref(d)) // 256))
    return t, d


# (operator, rows (of a shard), N, K, P, rank, weights as [n,k], tiles): 64x128 and 128x128 tiles of the float operators, and calls near them
@pytest.mark.parametrize("case", [("allreduce", 1000, 1544, 1234, 4, 0, False, "flexible 64x256"), ("allreduce", 650, 3332, 2310, 3, 0, True, "128x128"),
                                  ("allgather", 278, 4864, 4736, 2, 1, False, "128x128"), ("allreduce", 610, 4608, 5000, 8, 0, False, "flexible 64x256"),
                                  ("reduce_scatter", 1392, 1540, 2820, 8, 5, True, "128x128 dealt"), ("reduce_scatter", 600, 4104, 1032, 2, 1, False, "flexible 64x256"),
                                  ("allreduce", 644, 1492, 460, 3, 0, True, "64x128"), ("allreduce", 417, 2344, 808, 2, 0, False, "64x128"),
                                  ("allgather", 530, 464, 432, 4, 2, True, "64x128"), ("allgather", 600, 688, 760, 3, 0, False, "64x128"),
                                  ("allgather", 276, 776, 530, 16, 11, True, "128x128"), ("allgather", 431, 1104, 1090, 8, 4, False, "128x128")])
def test_float_larger_tiles(case):
    _need_gpu()
    op, m, N, K, P, rank, tb, kind = case
    g = torch.Generator(device="cuda:0").manual_seed(m)
    rand = lambda *shape: torch.randn(shape, device="cuda:0", generator=g)
    M = m * P if op == "allgather" else m
    A, B = rand(M, K).bfloat16(), (rand(K, N) * 0.05).bfloat16()
    Bd = B.T.contiguous() if tb else B
    rows = {"allreduce": m, "allgather": 0, "reduce_scatter": m // P}[op]
    peers = [rand(rows, N) for _ in range(P - 1)] if rows else []
    dump = torch.full((M, N), 7.0, device="cuda:0")
    if op == "allgather":
        shards = [s.contiguous() for s in A.split(m)]
        out = ops.allgather_matmul(shards[rank], shards[:rank] + shards[rank + 1:], Bd, rank, P, trans_b=tb, acc_dump=dump)
        got = dump
    elif op == "allreduce":
        out = ops.matmul_allreduce(A, Bd, peers, 0, P, trans_b=tb, acc_dump=dump)
        got = dump
    else:
        t, d = one_round(L.MATMUL_REDUCE_SCATTER, M, K, N, P, rank)
        ob = torch.full((L.load().catcoc_get_workspace_size(L.MATMUL_REDUCE_SCATTER, L.BF16, C.byref(t), C.byref(d)) // 4,), 3.0, device="cuda:0")
        out = ops.matmul_reduce_scatter(A, Bd, peers, rank, P, tiling=t, trans_b=tb, outbound=ob, acc_dump=dump, out=marked(rows, N, torch.bfloat16))
        tiles, full = ob.cpu().numpy().reshape(-1, 256), dump.cpu().numpy()
        for task, r, row, col, ws in tasks_of(L.MATMUL_REDUCE_SCATTER, t, d):
            if r != rank:
                r1, c1 = min(row + 128, (r + 1) * rows), min(col + 256, N)
                assert np.array_equal(tiles[ws:ws + r1 - row, :c1 - col], full[row:r1, col:c1]), task
        got = dump[rank * rows:(rank + 1) * rows]
    assert ran() == kind
    bound = 8 * K ** 0.5 * 2.0 ** -24 * torch.outer(A.double().norm(dim=1), B.double().norm(dim=0)) + 1e-9   # (as sum_bound)
    assert ((dump.double() - A.double() @ B.double()).abs() <= bound).all()
    for p in peers:
        got = got + p
    assert torch.equal(out, got.bfloat16())


# (rows per rank, N, K, P, rank, weights as [n,k], int32 peers): launches of 256x256 and 128x128 tiles; the kept rows (on small tiles) at the
# start, in the middle and at the end, k of whole pairs of steps and 4 to 124 bytes more, columns past a tile; one rank, whose kept rows are
# on tiles of both kinds
@pytest.mark.parametrize("case", [(335, 6912, 3204, 8, 5, False, False, "256x256 dealt"), (543, 3844, 3836, 8, 0, True, True, "256x256 dealt"),
                                  (664, 3460, 5888, 8, 7, True, False, "256x256 dealt"), (4344, 3844, 3836, 1, 0, True, False, "256x256"),
                                  (3700, 3840, 3072, 1, 0, False, False, "256x256")])
def test_quant_mixed_tiles(case):
    _need_gpu()
    rows, N, K, P, rank, tb, ri, kind = case
    M = rows * P
    g = torch.Generator(device="cuda:0").manual_seed(rows)
    x1, x2 = (torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda:0", generator=g) for shape in ((M, K), (K, N)))
    s1, s2 = (torch.empty(c, device="cuda:0").uniform_(0.001, 0.02, generator=g) for c in (M, N))
    b = torch.randint(-1000, 1000, (N,), dtype=torch.int32, device="cuda:0", generator=g)
    peers = [torch.randint(-2 ** 20, 2 ** 20, (rows, N), dtype=torch.int32, device="cuda:0", generator=g) if ri else torch.randn((rows, N), device="cuda:0", generator=g)
             for _ in range(P - 1)]
    t, d = one_round(L.QUANT_MATMUL_REDUCE_SCATTER, M, K, N, P, rank)
    size = L.load().catcoc_get_workspace_size(L.QUANT_MATMUL_REDUCE_SCATTER, L.INT8, C.byref(t), C.byref(d)) // 4
    ob = torch.full((size,), 3, dtype=torch.int32 if ri else torch.float32, device="cuda:0")
    dump, sums = torch.full((M, N), -7, dtype=torch.int32, device="cuda:0"), torch.full((rows, N), -7, dtype=torch.int32, device="cuda:0")
    out = ops.quant_matmul_reduce_scatter(x1, x2.T.contiguous() if tb else x2, s1, s2, b, peers, rank, P, tiling=t, trans_b=tb, reduce_int32=ri, outbound=ob,
                                          acc_dump=dump, c_accum=sums, out=marked(rows, N, torch.bfloat16))
    assert ran() == kind
    acc = (x1.double() @ x2.double()).to(torch.int32) + b   # (exact)
    kept = acc[rank * rows:(rank + 1) * rows]
    if ri:
        kept = kept + sum(peers)
    assert torch.equal(dump, acc) and torch.equal(sums, kept)
    deq = lambda a, sm: (a.float() * s2) * sm[:, None]
    want = deq(kept, s1[rank * rows:(rank + 1) * rows])
    for p in ([] if ri else peers):
        want = want + p
    assert torch.equal(out, want.bfloat16())
    full, tiles = (acc if ri else deq(acc, s1)), ob.reshape(-1, 256)
    for task, r, row, col, ws in tasks_of(L.QUANT_MATMUL_REDUCE_SCATTER, t, d):
        if r != rank:
            r1, c1 = min(row + 128, (r + 1) * rows), min(col + 256, N)
            assert torch.equal(tiles[ws:ws + r1 - row, :c1 - col], full[row:r1, col:c1]), task


@pytest.mark.parametrize("case", [("allgather", 845, 3940, 3330, 8, 3, True, "256x256"), ("allgather", 822, 2308, 6560, 8, 0, True, "256x256"),
                                  ("allreduce", 3438, 5892, 3712, 4, 0, True, "256x256"), ("reduce_scatter", 6184, 3072, 10752, 8, 2, False, "256x256 dealt"),
                                  ("reduce_scatter", 8144, 1696, 5120, 1, 0, True, "256x256"), ("reduce_scatter", 3000, 4096, 4096, 1, 0, False, "256x256")])
def test_float_mixed_tiles(case):
    test_float_larger_tiles(case)


# Two ranks' reduce-scatters (half of all rows kept, on small tiles) and k off the 16-byte grid, where flexible tiles ran before
@pytest.mark.parametrize("case", [(1513, 3584, 6280, 2, 1, False, False, "256x256 dealt"), (3978, 2048, 5604, 2, 0, True, True, "256x256 dealt")])
def test_quant_mixed_tiles_of_two_ranks(case):
    test_quant_mixed_tiles(case)


def test_float_mixed_tiles_off_the_16_byte_grid():
    test_float_larger_tiles(("allgather", 1024, 5120, 6148, 8, 3, False, "256x256"))


# Kept rows dealt out to the 128- and 64-row tiles: 16 or fewer to a tile (one group of a thread's rows; of 16 ranks more peers than fit at
# once), up to 32, up to 64 and as many as two ranks leave, tiles of unequal shares, first, last and a middle rank, columns past a tile; one rank, where none is dealt
@pytest.mark.parametrize("case", [(125, 4096, 1376, 8, 5, True, False, "128x128 dealt"), (65, 4096, 1040, 16, 15, False, True, "128x128 dealt"),
                                  (59, 4100, 1028, 16, 0, True, False, "64x128 dealt"), (123, 5116, 1660, 4, 1, True, False, "128x128 dealt"),
                                  (500, 4096, 1376, 2, 1, True, True, "128x128 dealt"), (103, 1792, 1732, 8, 3, False, False, "64x128 dealt"),
                                  (299, 544, 1280, 8, 7, True, False, "64x128 dealt"), (406, 2504, 496, 1, 0, True, False, "64x128"),
                                  (615, 1616, 1656, 1, 0, False, False, "64x128")])
def test_quant_dealt_rows(case):
    test_quant_mixed_tiles(case)


@pytest.mark.parametrize("case", [("reduce_scatter", 936, 6148, 1666, 8, 3, True, "flexible 128x256"),
                                  ("reduce_scatter", 1684, 2304, 520, 4, 0, False, "flexible 64x256"), ("reduce_scatter", 2400, 548, 1280, 16, 15, True, "64x128 dealt"),
                                  ("reduce_scatter", 480, 2344, 126, 8, 6, False, "64x128 dealt"), ("reduce_scatter", 510, 2344, 114, 2, 1, True, "64x128 dealt"),
                                  ("reduce_scatter", 1392, 1544, 1820, 8, 0, False, "128x128 dealt"), ("reduce_scatter", 1392, 1540, 1820, 4, 3, True, "128x128 dealt")])
def test_float_dealt_rows(case):
    test_float_larger_tiles(case)


# (rows, N, K, P, first kept row, kept rows, weights as [n,k]): sums of 128x128 blocks that several tiles add up: 32x32, 32x64, 64x64 and 64x128
# tiles, blocks of one tile and of few at the edges, blocks whose rows are all kept, negative and positive sums
@pytest.mark.parametrize("case", [(1, 132, 96, 2, 0, 1, True, "32x32", "64x128"), (33, 300, 1416, 8, 5, 7, False, "flexible 64x256", "flexible 64x256"),
                                  (128, 1280, 2416, 8, 0, 128, True, "32x32", "128x128"), (130, 516, 416, 4, 1, 128, True, "32x32", "128x128"),
                                  (300, 1408, 512, 8, 200, 40, True, "32x64", None), (80, 2784, 1060, 4, 60, 20, True, "32x64", "128x128"),
                                  (462, 1536, 2336, 4, 0, 116, True, "64x64", "128x128"), (409, 2688, 6232, 4, 300, 103, True, "64x128", "128x128")])
def test_quant_kept_rows_block_sums(case):
    _need_gpu()
    M, N, K, P, kb, kr, tb, *tiles = case
    g = torch.Generator(device="cuda:0").manual_seed(M + N)
    x1, x2 = (torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda:0", generator=g) for shape in ((M, K), (K, N)))
    x1[: M // 2] = x1[: M // 2].abs()   # (sums of either sign and size)
    x2[:, N // 2:] = x2[:, N // 2:].abs()
    s1, s2 = (torch.empty(c, device="cuda:0").uniform_(0.001, 0.02, generator=g) for c in (M, N))
    peers = [torch.randn((kr, N), device="cuda:0", generator=g) for _ in range(P - 1)]
    ws = torch.zeros(max(ops.splitk_plan(M, K, N, P, kb, kr)[0], 65536), dtype=torch.uint8, device="cuda:0")
    acc = (x1.double() @ x2.double()).to(torch.int64)
    others = acc.clone()
    others[kb:kb + kr] = 0
    want = torch.stack([others[r:r + 128, c:c + 128].sum() for r in range(0, M, 128) for c in range(0, N, 128)])
    out = None
    for w in (ws, ws, None):   # (the counter block is left at zero; without one the other kernels run)
        if w is None and tiles[1] is None:   # (needs one)
            continue
        cs = torch.full((want.numel(),), -7, dtype=torch.int64, device="cuda:0")
        got = ops.quant_matmul_splitk(x1, x2.T.contiguous() if tb else x2, s1, s2, None, peers, P, kb, kr, workspace=w, checksum=cs, trans_b=tb)
        assert ran() == tiles[0 if w is not None else 1]
        torch.cuda.synchronize()
        assert torch.equal(cs, want) and not ws[:65536].any()
        assert out is None or torch.equal(got, out)
        out = got
    y = (acc[kb:kb + kr].float() * s2) * s1[kb:kb + kr, None]
    for p in peers:
        y = y + p
    assert torch.equal(out, y.bfloat16())


# (rows, N, K, kept rows): up to 16 rows of a long k against few columns, on both sides of the line between the whole-k kernel and 32x32 tiles
@pytest.mark.parametrize("case", [(12, 640, 16384, 3, L.KERNEL_STREAMING), (16, 256, 14336, 4, L.KERNEL_STREAMING), (16, 128, 24576, 16, L.KERNEL_STREAMING), (8, 512, 12288, 2, L.KERNEL_STREAMING),
                                  (12, 672, 16384, 3, L.KERNEL_SMALL), (12, 512, 16384, 4, L.KERNEL_SMALL), (16, 256, 14208, 4, L.KERNEL_SMALL), (17, 512, 16384, 3, L.KERNEL_SMALL),
                                  (16, 128, 24448, 16, L.KERNEL_SMALL), (8, 512, 12288, 3, L.KERNEL_SMALL)])
def test_quant_few_rows_of_a_long_k(case):
    _need_gpu()
    M, N, K, kr, kernel = case
    g = torch.Generator(device="cuda:0").manual_seed(M + N)
    x1, x2 = (torch.randint(-127, 128, s, dtype=torch.int8, device="cuda:0", generator=g) for s in ((M, K), (N, K)))
    s1, s2 = (torch.empty(c, device="cuda:0").uniform_(0.001, 0.02, generator=g) for c in (M, N))
    peers = [torch.randn((kr, N), device="cuda:0", generator=g) for _ in range(7)]
    out = ops.quant_matmul_splitk(x1, x2, s1, s2, None, peers, 8, M - kr, kr, trans_b=True)
    assert L.last_launch().kernel == kernel
    y = ((x1[M - kr:].double() @ x2.T.double()).float() * s2) * s1[M - kr:, None]
    for p in peers:
        y = y + p
    assert torch.equal(out, y.bfloat16())


# (rows, N, K, P, first kept row, kept rows, weights as [n,k], int32 peers, checksums, tiles): the kept rows' int32 block from every tile, whole and in k
# slices; where the streaming kernels or flexible tiles would run k slices, whole small tiles are not taken
@pytest.mark.parametrize("case", [(46, 3360, 15872, 8, 40, 6, False, False, True, "32x32"), (129, 516, 648, 8, 128, 1, True, True, True, "32x32"),
                                  (8, 8192, 1024, 8, 0, 8, True, False, False, "32x32"), (300, 1284, 2416, 8, 260, 40, True, False, True, "32x64"),
                                  (203, 1376, 84, 3, 50, 70, True, True, False, "32x64"), (286, 1964, 124, 5, 0, 286, True, False, False, "64x64"),
                                  (336, 1696, 140, 3, 0, 336, False, True, False, "64x64"), (645, 2612, 1340, 2, 0, 300, True, True, True, "64x128"),
                                  (447, 2816, 1056, 4, 100, 112, False, False, False, "64x128"), (700, 4608, 1296, 2, 130, 300, False, True, False, "128x128"),
                                  (650, 4612, 1292, 3, 600, 50, True, False, True, "128x128"), (51, 1920, 12800, 4, 30, 13, True, False, True, "64x64/8"),
                                  (64, 512, 8192, 8, 0, 8, True, True, False, "32x32/8"), (67, 640, 4992, 8, 0, 67, False, False, False, "32x32/4"),
                                  (203, 4096, 1792, 8, 0, 203, True, False, False, "flexible 64x256/2"), (17, 384, 1344, 16, 3, 9, True, True, False, "streaming 128x128/4")])
def test_quant_kept_rows_int32_block(case):
    _need_gpu()
    M, N, K, P, kb, kr, tb, ri, with_sums, tiles = case
    g = torch.Generator(device="cuda:0").manual_seed(M + N)
    x1, x2 = (torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda:0", generator=g) for shape in ((M, K), (K, N)))
    s1, s2 = (torch.empty(c, device="cuda:0").uniform_(0.001, 0.02, generator=g) for c in (M, N))
    b = torch.randint(-1000, 1000, (N,), dtype=torch.int32, device="cuda:0", generator=g)
    peers = [torch.randint(-2 ** 20, 2 ** 20, (kr, N), dtype=torch.int32, device="cuda:0", generator=g) if ri else torch.randn((kr, N), device="cuda:0", generator=g)
             for _ in range(P - 1)]
    acc = (x1.double() @ x2.double()).to(torch.int64) + b
    others = acc.clone()
    others[kb:kb + kr] = 0
    sums = torch.stack([others[r:r + 128, c:c + 128].sum() for r in range(0, M, 128) for c in range(0, N, 128)])
    block = acc[kb:kb + kr].to(torch.int32) + (sum(peers) if ri else 0)
    y = (block.float() * s2) * s1[kb:kb + kr, None]
    for p in ([] if ri else peers):
        y = y + p
    ws = torch.zeros(max(ops.splitk_plan(M, K, N, P, kb, kr)[0], 65536), dtype=torch.uint8, device="cuda:0")
    cs = torch.full((sums.numel(),), -7, dtype=torch.int64, device="cuda:0") if with_sums else None
    ca = torch.full((kr + 1, N), -7, dtype=torch.int32, device="cuda:0")
    out = ops.quant_matmul_splitk(x1, x2.T.contiguous() if tb else x2, s1, s2, b, peers, P, kb, kr, workspace=ws, checksum=cs, c_accum=ca, trans_b=tb, reduce_int32=ri)
    assert ran() == tiles
    torch.cuda.synchronize()
    assert torch.equal(ca[:kr], block) and (ca[kr] == -7).all() and torch.equal(out, y.bfloat16()) and not ws[:65536].any()
    assert cs is None or torch.equal(cs, sums)


# (rows per rank, N, K, P): ragged rows or columns against [k,n] weights, of floats four k slices or more (test_ragged_launch_takes_the_slice_count_its_query_reports)
@pytest.mark.parametrize("case", [(145, 736, 2496, 2, "32x32"), (250, 640, 3776, 2, "32x64"), (284, 576, 3776, 4, "64x64"), (160, 544, 7232, 1, "32x32/3")])
def test_quant_ragged_slices_or_small_tiles(case):
    """Whole numbers: a caller's slice count and the library's small tiles leave the same bits."""
    _need_gpu()
    rows, N, K, P, tiles = case
    M, rank = rows * P, P - 1
    g = torch.Generator(device="cuda:0").manual_seed(M + N)
    x1, x2 = (torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda:0", generator=g) for shape in ((M, K), (K, N)))
    s1, s2 = (torch.empty(c, device="cuda:0").uniform_(0.001, 0.02, generator=g) for c in (M, N))
    peers = [torch.randn((rows, N), device="cuda:0", generator=g) for _ in range(P - 1)]
    t = ops.default_tiling(M, K, N, P, m0=0, n0=0, k0=0)
    d = L.make_desc(rank, P, [16] * (P - 1))
    size = L.load().catcoc_get_workspace_size(L.QUANT_MATMUL_REDUCE_SCATTER, L.INT8, C.byref(t), C.byref(d)) // 4
    need, f = ops.kslice_plan(L.QUANT_MATMUL_REDUCE_SCATTER, torch.int8, M, K, N, rank, P)
    assert f >= 4
    y = ((x1[rank * rows:].double() @ x2.double()).float() * s2) * s1[rank * rows:, None]
    for p in peers:
        y = y + p
    got = []
    for split_k, kind in ((0, tiles), (f, "flexible 64x256/%d" % f)):
        ws, ob = torch.zeros(need, dtype=torch.uint8, device="cuda:0"), torch.full((size,), 3.0, device="cuda:0")
        out = ops.quant_matmul_reduce_scatter(x1, x2, s1, s2, None, peers, rank, P, tiling=t, outbound=ob, workspace=ws, split_k=split_k)
        assert ran() == kind
        torch.cuda.synchronize()
        assert torch.equal(out, y.bfloat16())
        got.append(ob)
    assert torch.equal(got[0], got[1])


def sliced_workspace(need):
    """A workspace of more than the query asks for: counters at zero, marks behind what a launch may touch."""
    ws = torch.zeros(need + 4096, dtype=torch.uint8, device="cuda:0")
    ws[need:] = 0x5a
    return ws


def check_workspace(ws, need):
    assert not ws[:65536].any() and (ws[need:] == 0x5a).all() and ws[65536:need].any()   # (the last: slices ran)


# (operator, rows (of a shard), N, K, P, rank, weights as [n,k]): small tiles in k slices; k of odd chunks, rows and columns past a tile, more peers than
# registers hold at once, slices of unequal length
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", [("allreduce", 33, 896, 6656, 4, 0, False, "32x32/4"), ("allreduce", 7, 1024, 11262, 8, 0, True, "32x32/6"),
                                  ("allreduce", 20, 516, 8190, 16, 0, True, "32x32/8"), ("allgather", 2, 1536, 8448, 4, 3, True, "32x32/4"),
                                  ("allgather", 13, 1024, 14500, 8, 0, True, "32x64/4"), ("reduce_scatter", 44, 640, 6000, 2, 1, True, "32x32/6"),
                                  ("reduce_scatter", 112, 512, 6144, 4, 2, False, "32x32/4"), ("allreduce", 33, 1576, 5874, 8, 0, False, "64x64/8"),
                                  ("allreduce", 33, 1536, 6442, 3, 0, True, "64x64/8"), ("allreduce", 34, 2072, 3430, 8, 0, True, "32x64/3"),
                                  ("allreduce", 334, 304, 5808, 2, 0, False, "32x64/4")])
def test_float_k_slices(case, dtype):
    _need_gpu()
    op, m, N, K, P, rank, tb, kind = case
    g = torch.Generator(device="cuda:0").manual_seed(m)
    rand = lambda *shape: torch.randn(shape, device="cuda:0", generator=g)
    M = m * P if op == "allgather" else m
    A, B = rand(M, K).to(dtype), (rand(K, N) * 0.05).to(dtype)
    Bd = B.T.contiguous() if tb else B
    rows = {"allreduce": m, "allgather": 0, "reduce_scatter": m // P}[op]
    peers = [rand(rows, N) for _ in range(P - 1)] if rows else []
    comm = {"allreduce": L.MATMUL_ALLREDUCE, "allgather": L.ALLGATHER_MATMUL, "reduce_scatter": L.MATMUL_REDUCE_SCATTER}[op]
    need = ops.kslice_plan(comm, dtype, m, K, N, rank, P)[0]
    ws, first = sliced_workspace(need), None
    for _ in range(3):
        dump = torch.full((M, N), 7.0, device="cuda:0")
        if op == "allgather":
            shards = [s.contiguous() for s in A.split(m)]
            out = ops.allgather_matmul(shards[rank], shards[:rank] + shards[rank + 1:], Bd, rank, P, trans_b=tb, acc_dump=dump, workspace=ws)
            got = dump
        elif op == "allreduce":
            out = ops.matmul_allreduce(A, Bd, peers, 0, P, trans_b=tb, acc_dump=dump, workspace=ws)
            got = dump
        else:
            t, d = one_round(comm, M, K, N, P, rank)
            ob = torch.full((L.load().catcoc_get_workspace_size(comm, L.FP16, C.byref(t), C.byref(d)) // 4,), 3.0, device="cuda:0")
            out = ops.matmul_reduce_scatter(A, Bd, peers, rank, P, tiling=t, trans_b=tb, outbound=ob, acc_dump=dump, workspace=ws)
            tiles, full = ob.cpu().numpy().reshape(-1, 256), dump.cpu().numpy()
            for task, r, row, col, place in tasks_of(comm, t, d):
                if r != rank:
                    r1, c1 = min(row + 64, (r + 1) * rows), min(col + 256, N)
                    assert np.array_equal(tiles[place:place + r1 - row, :c1 - col], full[row:r1, col:c1]), task
            got = dump[rank * rows:(rank + 1) * rows]
        assert ran() == kind
        torch.cuda.synchronize()
        check_workspace(ws, need)
        assert first is None or torch.equal(first, dump)   # (slice order, whichever arrives last)
        first = dump
    bound = 8 * K ** 0.5 * 2.0 ** -24 * torch.outer(A.double().norm(dim=1), B.double().norm(dim=0)) + 1e-9   # (as sum_bound)
    assert ((dump.double() - A.double() @ B.double()).abs() <= bound).all()
    for p in peers:
        got = got + p
    assert torch.equal(out, got.to(dtype))


# (rows, N, K, P, first kept row, kept rows, weights as [n,k], int32 peers, dump): as above; of rows that are not kept only the sums, or all of them
@pytest.mark.parametrize("case", [(51, 1920, 12800, 4, 30, 13, True, False, False, "64x64/8"), (51, 1920, 12800, 4, 30, 13, True, False, True, "32x32/2"),
                                  (67, 640, 4992, 8, 0, 67, False, True, False, "32x32/4"), (134, 768, 4736, 8, 60, 17, False, False, False, "32x32/2"),
                                  (2, 512, 7680, 4, 1, 1, True, True, False, "32x32/6"), (24, 2560, 14848, 8, 21, 3, False, False, False, "32x32/3")])
def test_quant_k_slices(case):
    _need_gpu()
    M, N, K, P, kb, kr, tb, ri, with_dump, tiles = case
    g = torch.Generator(device="cuda:0").manual_seed(M + N)
    x1, x2 = (torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda:0", generator=g) for shape in ((M, K), (K, N)))
    s1, s2 = (torch.empty(c, device="cuda:0").uniform_(0.001, 0.02, generator=g) for c in (M, N))
    b = torch.randint(-1000, 1000, (N,), dtype=torch.int32, device="cuda:0", generator=g)
    peers = [torch.randint(-2 ** 20, 2 ** 20, (kr, N), dtype=torch.int32, device="cuda:0", generator=g) if ri else torch.randn((kr, N), device="cuda:0", generator=g)
             for _ in range(P - 1)]
    acc = (x1.double() @ x2.double()).to(torch.int64) + b
    others = acc.clone()
    others[kb:kb + kr] = 0
    sums = torch.stack([others[r:r + 128, c:c + 128].sum() for r in range(0, M, 128) for c in range(0, N, 128)])
    y = acc[kb:kb + kr].to(torch.int32) + (sum(peers) if ri else 0)
    y = (y.float() * s2) * s1[kb:kb + kr, None]
    for p in ([] if ri else peers):
        y = y + p
    need = ops.splitk_plan(M, K, N, P, kb, kr)[0]
    ws = sliced_workspace(need)
    for _ in range(3):
        cs = torch.full((sums.numel(),), -7, dtype=torch.int64, device="cuda:0")
        dump = torch.full((M, N), -7, dtype=torch.int32, device="cuda:0") if with_dump else None
        out = ops.quant_matmul_splitk(x1, x2.T.contiguous() if tb else x2, s1, s2, b, peers, P, kb, kr, workspace=ws, checksum=cs, acc_dump=dump, trans_b=tb, reduce_int32=ri)
        assert ran() == tiles
        torch.cuda.synchronize()
        check_workspace(ws, need)
        assert torch.equal(cs, sums) and torch.equal(out, y.bfloat16())
        assert dump is None or torch.equal(dump, acc.to(torch.int32))


# (rows per rank, N, K, P, rank, weights as [n,k], int32 peers): sums of tasks that several tiles add up: ranks of a few rows (many tasks to a tile), of a
# tile and a bit, of several task rows; columns that end in a task's first and second half; a long k (slices), 128-column tiles
@pytest.mark.parametrize("case", [(1, 256, 100, 8, 3, True, False, "32x32"), (2, 1000, 516, 16, 9, True, True, "32x32"), (5, 388, 1040, 8, 0, True, False, "32x32"),
                                  (33, 640, 416, 4, 3, False, True, "32x32"), (130, 900, 772, 2, 1, True, False, "32x64"),
                                  (8, 768, 15776, 2, 0, False, False, "32x32/8"), (69, 1024, 1024, 8, 5, True, False, "64x64"),
                                  (166, 768, 512, 8, 2, True, False, "64x64"), (219, 640, 9984, 8, 7, True, True, "64x128 dealt"),
                                  (300, 1800, 644, 4, 1, True, False, "flexible 128x256"), (88, 1984, 116, 8, 4, False, False, "64x128 dealt"),
                                  (43, 2192, 164, 16, 13, False, True, "64x128 dealt"), (96, 1984, 1504, 2, 1, False, False, "32x64"),
                                  (91, 1664, 1320, 4, 3, False, False, "64x64"), (184, 1440, 128, 8, 1, False, False, "128x128 dealt")])
def test_quant_task_sums(case):
    _need_gpu()
    rows, N, K, P, rank, tb, ri, tiles = case
    M = rows * P
    g = torch.Generator(device="cuda:0").manual_seed(rows)
    x1, x2 = (torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda:0", generator=g) for shape in ((M, K), (K, N)))
    x1[: M // 2] = x1[: M // 2].abs()
    x2[:, N // 2:] = x2[:, N // 2:].abs()
    s1, s2 = (torch.empty(c, device="cuda:0").uniform_(0.001, 0.02, generator=g) for c in (M, N))
    b = torch.randint(-1000, 1000, (N,), dtype=torch.int32, device="cuda:0", generator=g)
    peers = [torch.randint(-2 ** 20, 2 ** 20, (rows, N), dtype=torch.int32, device="cuda:0", generator=g) if ri else torch.randn((rows, N), device="cuda:0", generator=g)
             for _ in range(P - 1)]
    t, d = one_round(L.QUANT_MATMUL_REDUCE_SCATTER, M, K, N, P, rank)
    tasks = list(tasks_of(L.QUANT_MATMUL_REDUCE_SCATTER, t, d))
    acc = ((x1.double() @ x2.double()).to(torch.int64) + b).cpu()
    step = 64 if rows <= 64 else 128
    want = torch.full((len(tasks),), 77, dtype=torch.int64)
    for task, r, row, col, ws in tasks:
        if r != rank:
            want[task] = acc[row:min(row + step, (r + 1) * rows), col:min(col + 256, N)].sum()
    kept = acc[rank * rows:(rank + 1) * rows].to(torch.int32).to("cuda:0")
    y = ((kept + sum(peers) if ri else kept).float() * s2) * s1[rank * rows:(rank + 1) * rows, None]
    for p in ([] if ri else peers):
        y = y + p
    need = ops.kslice_plan(L.QUANT_MATMUL_REDUCE_SCATTER, L.INT8, M, K, N, rank, P, tiling=t)[0]
    ws = torch.zeros(max(need, 65536), dtype=torch.uint8, device="cuda:0")
    for w in (ws, ws, None):   # (without counters sums are not small tiles')
        cs = torch.full((len(tasks),), 77, dtype=torch.int64, device="cuda:0")
        out = ops.quant_matmul_reduce_scatter(x1, x2.T.contiguous() if tb else x2, s1, s2, b, peers, rank, P, tiling=t, trans_b=tb, reduce_int32=ri, checksum=cs, workspace=w)
        assert ran() == tiles if w is not None else L.last_launch().kernel != L.KERNEL_SMALL
        torch.cuda.synchronize()
        assert torch.equal(cs.cpu(), want) and torch.equal(out, y.bfloat16()) and not ws[:65536].any()


def test_small_tiles_replay_from_a_hip_graph():
    """A block-sum call, a sliced one and a task-sum one on one workspace in a captured graph: every replay, on new inputs and with eager calls in
    between, gives what an eager call gives."""
    _need_gpu()
    g = torch.Generator(device="cuda:0").manual_seed(5)
    i8 = lambda *s: torch.randint(-127, 128, s, dtype=torch.int8, device="cuda:0", generator=g)
    ws = torch.zeros(32 << 20, dtype=torch.uint8, device="cuda:0")
    s1, s2 = torch.full((400,), 0.01, device="cuda:0"), torch.full((1024,), 0.02, device="cuda:0")
    x1, x2 = i8(51, 12800), i8(768, 12800)
    y1, y2 = i8(400, 1024), i8(1024, 1024)
    peers = [torch.randn((13, 768), device="cuda:0", generator=g) for _ in range(3)]
    more = [torch.randn((50, 1024), device="cuda:0", generator=g) for _ in range(7)]
    t, d = one_round(L.QUANT_MATMUL_REDUCE_SCATTER, 400, 1024, 1024, 8, 3)
    tasks = len(list(tasks_of(L.QUANT_MATMUL_REDUCE_SCATTER, t, d)))

    def calls(o):
        ops.quant_matmul_splitk(x1, x2, s1[:51], s2[:768], None, peers, 4, 30, 13, workspace=ws, checksum=o[1], out=o[0], trans_b=True)
        ops.quant_matmul_reduce_scatter(y1, y2, s1, s2, None, more, 3, 8, tiling=t, trans_b=True, checksum=o[3], out=o[2], workspace=ws)
        ops.quant_matmul_splitk(y1[:100], y2, s1[:100], s2, None, [more[0][:9]], 2, 60, 9, workspace=ws, checksum=o[5], out=o[4], trans_b=True)

    def outputs():
        z = lambda *s, **k: torch.zeros(s, device="cuda:0", **k)
        return [z(13, 768, dtype=torch.bfloat16), z(6, dtype=torch.int64), z(50, 1024, dtype=torch.bfloat16), z(tasks, dtype=torch.int64), z(9, 1024, dtype=torch.bfloat16), z(8, dtype=torch.int64)]

    captured, eager = outputs(), outputs()
    calls(captured)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        calls(captured)
    for i in range(4):
        x1.copy_(i8(51, 12800))
        y2.copy_(i8(1024, 1024))
        calls(eager)
        for o in captured:
            o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(captured, eager)) and captured[1].any() and captured[3].any() and not ws[:65536].any(), i


# (rows per rank, N, K, P, rank, weights as [n,k]): as test_quant_task_sums; sums of floats are added in one order
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", [(1, 256, 100, 8, 3, True, "32x32"), (5, 388, 1040, 8, 0, True, "32x32"), (33, 640, 416, 4, 3, False, "32x32"),
                                  (130, 900, 772, 2, 1, True, "32x64"), (37, 1024, 12672, 4, 2, False, "flexible 64x256/17"), (43, 1920, 1152, 2, 0, True, "32x32"),
                                  (363, 640, 2364, 8, 6, False, "64x128 dealt"), (301, 1800, 646, 4, 1, True, "128x128 dealt"), (72, 1000, 94, 8, 2, False, "64x64"),
                                  (85, 836, 4584, 4, 2, True, "64x64/3"), (24, 1312, 5824, 4, 0, False, "32x64/4"), (264, 1104, 128, 8, 1, False, "128x128 dealt")])
def test_float_task_sums(case, dtype):
    _need_gpu()
    rows, N, K, P, rank, tb, tiles = case
    M = rows * P
    g = torch.Generator(device="cuda:0").manual_seed(rows)
    A, B = torch.randn((M, K), device="cuda:0", generator=g).to(dtype), (torch.randn((K, N), device="cuda:0", generator=g) * 0.05).to(dtype)
    Bd = B.T.contiguous() if tb else B
    peers = [torch.randn((rows, N), device="cuda:0", generator=g) for _ in range(P - 1)]
    comm = L.MATMUL_REDUCE_SCATTER
    t, d = one_round(comm, M, K, N, P, rank)
    tasks = list(tasks_of(comm, t, d))
    step = 64 if rows <= 64 else 128
    need = ops.kslice_plan(comm, dtype, M, K, N, rank, P, tiling=t)[0]
    ws = torch.zeros(max(need, 65536), dtype=torch.uint8, device="cuda:0")
    first = None
    for _ in range(4):
        cs, dump = torch.full((len(tasks),), 77.0, dtype=torch.float64, device="cuda:0"), torch.zeros((M, N), device="cuda:0")
        out = ops.matmul_reduce_scatter(A, Bd, peers, rank, P, tiling=t, trans_b=tb, checksum=cs, acc_dump=dump, workspace=ws)
        assert ran() == tiles
        torch.cuda.synchronize()
        assert not ws[:65536].any() and (first is None or torch.equal(first, cs))
        first = cs
    bound = 8 * K ** 0.5 * 2.0 ** -24 * torch.outer(A.double().norm(dim=1), B.double().norm(dim=0)) + 1e-9   # (as sum_bound)
    assert ((dump.double() - A.double() @ B.double()).abs() <= bound).all()
    full, got = dump.double().cpu(), cs.cpu()
    for task, r, row, col, _ in tasks:
        own = full[row:min(row + step, (r + 1) * rows), col:min(col + 256, N)]
        assert got[task] == 77.0 if r == rank else abs(got[task] - own.sum()) <= own.numel() * 2.0 ** -51 * own.abs().sum(), task
    y = dump[rank * rows:(rank + 1) * rows]
    for p in peers:
        y = y + p
    assert torch.equal(out, y.to(dtype))


# (rows, N, K, P, first kept row or rank, kept rows or 0: a reduce-scatter's, weights as [n,k]): sums of W8A8 tiles in k slices under a bias at either end of
# its range: the whole accumulators are the bias itself, a slice's own sum and the bias are past the end
@pytest.mark.parametrize("case", [(64, 512, 8192, 8, 20, 8, True, "32x32/8"), (70, 384, 8192, 2, 69, 1, False, "32x32/6"), (16, 768, 15776, 2, 0, 0, False, "32x32/8"),
                                  (40, 512, 8192, 4, 3, 0, True, "32x32/6")])
def test_sums_of_k_slices_with_a_bias_at_the_end_of_its_range(case):
    _need_gpu()
    M, N, K, P, at, kr, tb, tiles = case
    g = torch.Generator(device="cuda:0").manual_seed(M + N)
    u, v = (torch.randint(90, 128, shape, dtype=torch.int8, device="cuda:0", generator=g) for shape in ((M, K // 2), (K // 2, N)))
    up = torch.arange(N, device="cuda:0") % 3 != 0   # (more of one sign: what the two kinds of columns are off by does not cancel)
    v = torch.where(up, v, -v)
    x1, x2 = torch.cat([u, u], 1), torch.cat([v, -v], 0)
    b = torch.randint(0, 1000, (N,), dtype=torch.int32, device="cuda:0", generator=g)
    b = torch.where(up, 2 ** 31 - 1 - b, -2 ** 31 + b)
    s1, s2 = (torch.empty(c, device="cuda:0").uniform_(0.001, 0.02, generator=g) for c in (M, N))
    acc = b.to(torch.int64).expand(M, N)
    rows, first = (kr, at) if kr else (M // P, at * (M // P))
    peers = [torch.randn((rows, N), device="cuda:0", generator=g) for _ in range(P - 1)]
    y = (b.float() * s2) * s1[first:first + rows, None]
    for p in peers:
        y = y + p
    x2d = x2.T.contiguous() if tb else x2
    if kr:
        need = ops.splitk_plan(M, K, N, P, at, kr)[0]
        others = acc.clone()
        others[first:first + rows] = 0
        want = torch.stack([others[r:r + 128, c:c + 128].sum() for r in range(0, M, 128) for c in range(0, N, 128)]).cpu()
        run = lambda cs, ws: ops.quant_matmul_splitk(x1, x2d, s1, s2, b, peers, P, at, kr, workspace=ws, checksum=cs, trans_b=tb)
    else:
        t, d = one_round(L.QUANT_MATMUL_REDUCE_SCATTER, M, K, N, P, at)
        need = ops.kslice_plan(L.QUANT_MATMUL_REDUCE_SCATTER, L.INT8, M, K, N, at, P, tiling=t)[0]
        tasks = list(tasks_of(L.QUANT_MATMUL_REDUCE_SCATTER, t, d))
        want = torch.full((len(tasks),), 77, dtype=torch.int64)
        for task, r, row, col, _ in tasks:
            if r != at:
                want[task] = acc[row:min(row + 64, (r + 1) * rows), col:min(col + 256, N)].sum()
        run = lambda cs, ws: ops.quant_matmul_reduce_scatter(x1, x2d, s1, s2, b, peers, at, P, tiling=t, trans_b=tb, checksum=cs, workspace=ws)
    ws = sliced_workspace(need)
    cs = torch.full((want.numel(),), 77, dtype=torch.int64, device="cuda:0")
    out = run(cs, ws)
    assert ran() == tiles
    torch.cuda.synchronize()
    check_workspace(ws, need)
    assert torch.equal(out, y.bfloat16()) and torch.equal(cs.cpu(), want)


# (rows, N, K, P, rank, weights as [n,k], workspace, tiles without and with a choice: floats, W8A8): what a caller says about halves of kept tiles changes no
# bit, whichever tiles run: small and mixed ones, in k slices, whole flexible tiles or aligned ones instead, flexible ones in k slices
@pytest.mark.parametrize("kind", [torch.float16, torch.bfloat16, torch.int8])
@pytest.mark.parametrize("case", [(2048, 2048, 1792, 8, 3, False, False, "128x128 dealt", "128x128 dealt", "128x128 dealt", "128x128 dealt"),
                                  (1024, 512, 512, 8, 7, True, False, "32x64", "32x64", "32x64", "32x64"),
                                  (4096, 4096, 1792, 8, 2, True, False, "256x256 dealt", "256x256 dealt", "256x256 dealt", "256x256 dealt"),
                                  (512, 512, 6144, 4, 2, False, True, "32x64/2", "32x64/2", "32x32", "32x32"),
                                  (512, 4096, 1024, 4, 1, True, False, "64x128 dealt", "64x128 dealt", "64x128 dealt", "64x128 dealt"),
                                  (1024, 1024, 8192, 2, 0, True, True, "64x64", "64x64", "64x64", "64x64"),
                                  (512, 8192, 512, 2, 1, True, True, "flexible 64x256", "aligned 128x256", "aligned 128x256", "aligned 128x256"),
                                  (512, 1024, 8192, 2, 1, False, True, "flexible 64x256/8", "flexible 64x256/8", "flexible 64x256/6", "flexible 64x256/6")])
def test_halves_of_kept_tiles_change_no_bit(case, kind):
    _need_gpu()
    M, N, K, P, rank, tb, slices, *tiles = case
    g = torch.Generator(device="cuda:0").manual_seed(M + K)
    quant = kind == torch.int8
    if quant:
        a, b = (torch.randint(-127, 128, s, dtype=torch.int8, device="cuda:0", generator=g) for s in ((M, K), (N, K) if tb else (K, N)))
    else:
        a, b = torch.randn((M, K), device="cuda:0", generator=g).to(kind), (torch.randn((N, K) if tb else (K, N), device="cuda:0", generator=g) * 0.05).to(kind)
    s1, s2 = (torch.empty(c, device="cuda:0").uniform_(0.001, 0.02, generator=g) for c in (M, N))
    peers = [torch.randn((M // P, N), device="cuda:0", generator=g) for _ in range(P - 1)]
    comm = L.QUANT_MATMUL_REDUCE_SCATTER if quant else L.MATMUL_REDUCE_SCATTER
    t, d = one_round(comm, M, K, N, P, rank)
    size = L.load().catcoc_get_workspace_size(comm, L.INT8 if quant else L.FP16, C.byref(t), C.byref(d)) // 4
    need = max(ops.kslice_plan(comm, kind, M, K, N, rank, P, tiling=t)[0], 65536)
    results = []
    for choice in (None, False, True, "kept-only"):
        ob, dump = torch.full((size,), 3.0, device="cuda:0"), torch.zeros((M, N), dtype=torch.int32 if quant else torch.float32, device="cuda:0")
        kw = dict(tiling=t, trans_b=tb, outbound=ob, acc_dump=dump, kept_split=choice, workspace=torch.zeros(need, dtype=torch.uint8, device="cuda:0") if slices else None)
        out = ops.quant_matmul_reduce_scatter(a, b, s1, s2, None, peers, rank, P, **kw) if quant else ops.matmul_reduce_scatter(a, b, peers, rank, P, **kw)
        assert ran() == tiles[2 * quant + (choice in (False, True))]
        torch.cuda.synchronize()
        results.append((out, dump, ob))
    for r in results[1:]:
        assert all(torch.equal(x, y) for x, y in zip(r, results[0]))


# (rows, N, K, weights as [n,k], k slices): 32x32, 32x64, 64x64 tiles, whole and in k slices, 64x128 and 128x128 ones
@pytest.mark.parametrize("case", [(100, 2048, 1024, True, False, "32x32"), (512, 1024, 1024, False, False, "32x64"), (1000, 512, 2052, True, False, "32x64"),
                                  (96, 512, 8192, True, True, "32x32/4"), (300, 1032, 6148, True, True, "64x64/3"), (650, 3332, 2310, True, False, "128x128")])
def test_equal_rows_have_equal_sums_wherever_they_lie(case):
    _need_gpu()
    M, N, K, tb, slices, tiles = case
    g = torch.Generator(device="cuda:0").manual_seed(M)
    A = torch.randn((1, K), device="cuda:0", generator=g).bfloat16().expand(M, K).contiguous()
    B = torch.randn((N, K) if tb else (K, N), device="cuda:0", generator=g).bfloat16()
    need = ops.kslice_plan(L.MATMUL_ALLREDUCE, torch.bfloat16, M, K, N, 0, 2)[0]
    dump = torch.zeros((M, N), device="cuda:0")
    ops.matmul_allreduce(A, B, [torch.zeros((M, N), device="cuda:0")], 0, 2, trans_b=tb, acc_dump=dump, workspace=torch.zeros(need, dtype=torch.uint8, device="cuda:0") if slices else None)
    assert ran() == tiles
    torch.cuda.synchronize()
    assert torch.equal(dump, dump[:1].expand(M, N))


# 128-column tiles of 96, 160 and 192 rows: both layouts of the weights, rows, columns and k past a tile, a chunk and a 16-byte piece, dealt and consecutive rows
@pytest.mark.parametrize("case", [(66, 5088, 616, 8, 7, False, False, "96x128 dealt"), (171, 1824, 808, 8, 0, True, True, "96x128 dealt"),
                                  (306, 3392, 528, 4, 3, False, False, "160x128 dealt"), (158, 3328, 556, 8, 5, True, True, "160x128 dealt"),
                                  (171, 3744, 568, 8, 5, False, True, "192x128 dealt"), (266, 4768, 544, 4, 3, True, False, "192x128 dealt")])
def test_quant_rows_between(case):
    test_quant_mixed_tiles(case)


@pytest.mark.parametrize("case", [("allreduce", 630, 3680, 552, 2, 0, True, "96x128"), ("allgather", 637, 1568, 646, 2, 0, True, "96x128"),
                                  ("reduce_scatter", 640, 4480, 894, 8, 4, False, "96x128 dealt"), ("allreduce", 586, 7680, 606, 2, 0, True, "160x128"),
                                  ("allgather", 366, 6304, 564, 2, 1, True, "160x128"), ("reduce_scatter", 880, 5056, 668, 8, 2, False, "160x128 dealt"),
                                  ("allgather", 95, 7424, 512, 8, 4, True, "192x128"), ("reduce_scatter", 1240, 4416, 524, 8, 2, True, "192x128 dealt")])
def test_float_rows_between(case):
    test_float_larger_tiles(case)


@pytest.mark.parametrize("case", [(171, 1952, 556, 8, 2, False, True, "96x128 dealt"), (159, 3392, 524, 8, 4, False, False, "160x128 dealt"),
                                  (117, 5440, 536, 8, 4, True, True, "192x128 dealt")])
def test_quant_task_sums_rows_between(case):
    test_quant_task_sums(case)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("case", [(334, 1696, 794, 4, 3, False, "96x128 dealt"), (132, 4288, 624, 8, 4, False, "160x128 dealt"), (141, 4768, 514, 8, 1, True, "192x128 dealt")])
def test_float_task_sums_rows_between(case, dtype):
    test_float_task_sums(case, dtype)


# Explicit kept rows on tiles of 96, 160 and 192 rows: kept rows that end inside a tile, all rows, nine ranks
@pytest.mark.parametrize("case", [(335, 5472, 544, 8, 62, 270, False, False, "96x128"), (323, 5536, 540, 8, 0, 323, True, True, "96x128"),
                                  (773, 5024, 516, 9, 169, 602, False, False, "160x128"), (657, 5824, 512, 2, 115, 295, True, True, "160x128"),
                                  (862, 5664, 520, 4, 309, 433, False, True, "192x128"), (837, 5568, 528, 8, 178, 438, True, False, "192x128")])
def test_quant_kept_rows_on_rows_between(case):
    test_quant_kept_rows(case)


# Calls beside which other kernels are slower, or that were slower on others: large and small tiles that fill the CUs exactly once; checksums on
# flexible tiles; k slices of a decode call as [k,n]
def test_mixed_tiles_that_fill_the_cus_once():
    test_float_larger_tiles(("reduce_scatter", 1800, 5888, 1344, 8, 3, False, "256x256 dealt"))
    assert L.last_launch().largeTiles == 161   # (and 92 of 128x128)


def test_checksums_on_flexible_tiles_beside_small_ones():
    test_quant_task_sums((565, 1440, 784, 8, 3, False, False, "flexible 128x256"))


def test_k_slices_beside_small_tiles():
    test_quant_kept_rows((388, 512, 7936, 8, 0, 388, False, False, "flexible 64x256/9"))
