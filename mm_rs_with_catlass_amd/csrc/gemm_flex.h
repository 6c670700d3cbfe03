// Tiles that need not line up with the schedule's tiles, and the epilogue that goes with them.
//
// A launch of the direct-to-LDS kernels in flexible mode (FX) cuts the rows of the whole problem -- all ranks' rows behind
// each other -- into row tiles of its own, whatever the ranks' boundaries, and lets the row decide in the epilogue where its
// values go: to the kept rows (peers added), to its place in the tile-linear workspace, or into its task's checksum.  With
// eight ranks of 125 rows that is 8 tiles of 128 rows and not 8 tiles plus their edges, with eight ranks of 8 rows one tile
// and not eight, and the shards of an all-gather share tiles in the same way.  Rows past the end repeat the last row on
// the way in and are dropped on the way out; so are columns.
//
// The epilogue goes through LDS once (32 rows of a wave at a time), after which a lane holds four consecutive columns of a
// row: every access to peers, output, workspace and dumps is 8 or 16 bytes per lane over whole row segments, and what a
// row is to do is one table entry per row.
//
// Bound by the same things as the aligned kernels it shares its main loop with: the tile copies and the matrix pipes for long
// k, the peers' stream for short k.  Measured against what ran these launches before (a kernel that staged its tiles through
// registers, or one thread per output element), launches alternating: fp16 all-gather 8 x [1024,6148] x [6148,5120]
// 243 ms -> 0.522 ms = 988 TFLOP/s (12296-byte rows, 8 bytes of k left over), W8A8 64x8192x8192 with 8 rows kept 22.7 -> 19.9 us.
// Smaller launches are small tiles' (gemm_few.h, gemm_mid.h): W8A8 reduce-scatter 1000x1376x4096 of eight ranks, stored tiles, took 277 us
// before either, bf16 all-reduce 16x1024x8192 28.7.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "gemm_fused_kernel.h"

namespace catcoc {

// ---- launch position -> tile ------------------------------------------------------------------------------------------
struct FlexTile {
    uint32_t row0, rowsValid;   // global rows (of all ranks) [row0, row0 + rowsValid)
    uint32_t col0, colsValid;
    uint32_t index;             // rowTile * colTiles + colTile
};

CATCOC_HD uint32_t flex_row_start(const GemmArgs &a, uint32_t rt, uint32_t &valid)
{
    const FlexParams &f = a.fx;
    if (f.perRank) {   // one schedule tile row per row tile: checksums of tasks that are not whole ranks
        const uint32_t rank = rt / a.sched.loopsM, mi = rt - rank * a.sched.loopsM;
        valid = umin(a.sched.m0, a.sched.mRank - mi * a.sched.m0);
        return rank * a.sched.mRank + mi * a.sched.m0;
    }
    const uint32_t row0 = rt * f.rowStep;
    valid = umin(f.rowStep, f.rows - row0);
    return row0;
}

// Consecutive workgroups go round-robin to the eight XCDs, each with an L2 of its own: XCD x takes the x-th contiguous
// eighth of the tile sequence, and the sequence walks bands of eight tile rows, so that the tiles in flight on one XCD form
// a compact block of the grid.  Row tiles with kept rows of a reduce-scatter launch come first (their epilogue streams the
// peers' partials: the longest chain of the launch), dealt to the XCDs in the same way.
CATCOC_HD uint32_t xcd_eighth(uint32_t pos, uint32_t count)
{
    const uint32_t x = pos & 7u, q = count >> 3, r = count & 7u;
    return x * q + umin(x, r) + (pos >> 3);
}

CATCOC_HD void flex_tile(const GemmArgs &a, uint32_t pos, FlexTile &t, uint32_t &slice)
{
    const FlexParams &f = a.fx;
    const uint32_t first = f.slices > 1 ? 0u : f.keptTiles * f.colTiles;
    const bool kept = pos < first;
    uint32_t seq, rows;
    slice = 0;
    if (f.slices > 1) {   // an XCD takes neighbouring tiles of the same k slice: they share its rows of A; no tile is longer than another
        const uint32_t tiles = f.rowTiles * f.colTiles;
        seq = xcd_eighth(pos, tiles * f.slices);
        slice = seq / tiles;
        seq -= slice * tiles;
        rows = f.rowTiles;
    } else if (kept) { rows = f.keptTiles; seq = xcd_eighth(pos, first); }
    else { rows = f.rowTiles - f.keptTiles; seq = xcd_eighth(pos - first, rows * f.colTiles); }
    const uint32_t BAND = 8u;
    const uint32_t band = seq / (BAND * f.colTiles), in = seq - band * (BAND * f.colTiles);
    const uint32_t w = umin(BAND, rows - band * BAND);
    const uint32_t ct = in / w;
    uint32_t rt = band * BAND + (in - ct * w);
    if (kept) rt += f.keptTile0;
    else if (f.slices <= 1 && rt >= f.keptTile0) rt += f.keptTiles;
    t.row0 = flex_row_start(a, rt, t.rowsValid);
    t.col0 = ct * 256u;
    t.colsValid = umin(256u, a.N - t.col0);
    t.index = rt * f.colTiles + ct;
}

// ---- a row's place ------------------------------------------------------------------------------------------------------
// Row `ri` of rank `r` in column tile `ni`: its task, and its row of the tile-linear workspace (tile_sched.h: task_tile).
__device__ __forceinline__ void flex_task_of(const SchedParams &s, uint32_t r, uint32_t ri, uint32_t ni, uint32_t &task, uint32_t &wsRow)
{
    const uint32_t mi = ri / s.m0;
    const uint32_t inRank = swizzle_block_index(s.off, s.dir, s.loopsM, s.loopsN, mi, ni);
    const uint32_t perRank = s.blockPerComm / s.P;
    const uint32_t round = inRank / perRank, idx = inRank - round * perRank;
    const uint32_t commLoops = ceil_div(s.coreLoops, s.blockPerComm);
    const uint32_t actual = (round == commLoops - 1u) ? s.coreLoops - round * s.blockPerComm : s.blockPerComm;
    const uint32_t b = r * (actual / s.P) + idx;
    task = round * s.blockPerComm + b;
    wsRow = ((round % s.stages) * s.blockPerComm + b) * s.m0 + (ri - mi * s.m0);
}

// Row of the problem that row v of the flexible tiles is: behind the hole that a mixed launch (eight waves, 256-row tiles) leaves to its small
// tiles.  (The other launches have none, and the two arguments are a trip to host memory: 0.3 us of 26.)
template <bool HOLE>
CATCOC_HD uint32_t flex_row(const GemmArgs &a, uint32_t v) { return HOLE && a.fx.holeRows != 0 && v >= a.fx.hole0 ? v + a.fx.holeRows : v; }

// Address of row v of the left operand (all-gather: row v of the shards behind each other).
__device__ __forceinline__ const unsigned char *flex_row_ptr(const GemmArgs &a, uint32_t v, int64_t ldaB)
{
    if (a.sched.op == OP_ALLGATHER) {
        uint32_t in;
        const uint32_t r = fast_div(v, a.fx.dRank, in);
        return (const unsigned char *)a.a[r] + (size_t)in * ldaB;
    }
    return (const unsigned char *)a.a[0] + (size_t)v * ldaB;
}

// 16 bytes from p of which the first `valid` exist (a multiple of four; zero or less: none), the rest as zeros.  A word that
// does not exist is read at `last` instead, the offset from p of a word of the same row that does (it may be negative): no
// branches, so the loads of all pieces of a thread are in flight together.  4-byte aligned.
__device__ __forceinline__ v4i load16_guarded(const unsigned char *p, int valid, int last)
{
    v4i v;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const int at = 4 * d < last ? 4 * d : last;   // (last = offset from p of the last word that exists; may be negative)
        const int x = *(const int *)(p + at);
        v[d] = 4 * d < valid ? x : 0;
    }
    return v;
}

// ---- epilogue -------------------------------------------------------------------------------------------------------------
enum : uint32_t { FX_SKIP = 0u, FX_KEPT = 1u << 30, FX_OUT = 2u << 30, FX_SUM = 3u << 30, FX_KIND = 3u << 30, FX_INDEX = (1u << 30) - 1u };

constexpr int FLEX_STAGING = 4 * 16384;                 // one 16 KiB area per wave
constexpr int FLEX_POOL = FLEX_STAGING + 128 * 8 + 16 * 8 * 8 + 16 * 4;   // + the row table + the sums of up to 16 tasks, per half wave
constexpr int FLEX_POOL8 = 160 * 1024;   // of eight waves and 256 rows (mixed launches): the rings, all of the LDS
static_assert(2 * FLEX_STAGING + 256 * 8 + 16 * 16 * 8 + 16 * 4 <= FLEX_POOL8, "the epilogue of eight waves fits");

// Sums over lanes, always in the same order: cross-lane adds in the vector unit (a shuffle is a trip through the LDS unit).
template <int CTRL, int ROWS, typename T>
__device__ __forceinline__ T dpp_add64(T v)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
    return v + __builtin_bit_cast(T, ((unsigned long long)(uint32_t)hi << 32) | (uint32_t)lo);
}
// over each half of a wave, in its last lane
template <typename T>
__device__ __forceinline__ T half_sum64(T v)
{
    v = dpp_add64<0x111, 0xf>(v);   // row_shr:1, 2, 4, 8: lane 15 of every row of 16 holds the row's sum
    v = dpp_add64<0x112, 0xf>(v);
    v = dpp_add64<0x114, 0xf>(v);
    v = dpp_add64<0x118, 0xf>(v);
    return dpp_add64<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
}
// over the 64 lanes, in lane 63
template <typename T>
__device__ __forceinline__ T wave_sum64(T v)
{
    return dpp_add64<0x143, 0xc>(half_sum64(v));   // row_bcast:31 into rows 2 and 3
}

// A wave's rows [32 * mb, +32) of its 128 columns into its staging area: rows of 512 bytes, 16-byte piece c of row r at c * 16 ^ flex_turn(r), which
// keeps what is written together in different banks.  acc[mb][nb][r] of 32x32 MFMAs is row mb*32 + (r>>2)*8 + (lane>>5)*4 + (r&3), column nb*32 +
// (lane&31); acc[i][j][r] of 16x16 ones (L16) row i*16 + (lane>>4)*4 + r, column j*16 + (lane&15).  What follows reads other lanes' values: the LDS
// unit keeps a wave's accesses in order, the compiler is told by the empty asm statements.
template <bool L16>
__device__ __forceinline__ uint32_t flex_turn(uint32_t row) { return L16 ? ((row >> 2) & 3u) << 6 : ((row >> 2) & 1u) << 7; }

template <bool L16, typename Acc>
__device__ __forceinline__ void flex_stage(const Acc &acc, int mb, unsigned char *st, uint32_t lane)
{
    asm volatile("" ::: "memory");
    if constexpr (L16) {
        const uint32_t l16 = lane & 15, quad = lane >> 4;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const auto e = acc[2 * mb + i][j][r];
                    *(int *)(st + (i * 16 + quad * 4 + r) * 512 + (((j * 16 + l16) * 4) ^ (quad << 6))) = __builtin_bit_cast(int, e);
                }
    } else {
        const uint32_t c32 = lane & 31, h = lane >> 5;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint32_t wrow = (r >> 2) * 8 + h * 4 + (r & 3);
#pragma unroll
            for (int nb = 0; nb < 4; ++nb) {
                const auto e = acc[mb][nb][r];
                *(int *)(st + wrow * 512 + (((nb * 32 + c32) * 4) ^ (h << 7))) = __builtin_bit_cast(int, e);
            }
        }
    }
    asm volatile("" ::: "memory");
}

// Wave (wm, wn) has rows wm*32*MB and columns wn*128 of the tile.  NW waves, two of them side by side: tiles of 16 * MB * NW rows.
template <uint32_t DT, int MB, int NW, bool L16, typename Acc>
__device__ __forceinline__ void flex_epilogue(const GemmArgs &args, const Acc &acc, unsigned char *smem, const FlexTile &t)
{
    constexpr bool I8 = DT == DT_I8;
    constexpr uint32_t ROWS = 16u * MB * NW, TABLE = NW == 4 ? 128u : ROWS;
    using Sum = typename std::conditional<I8, long long, double>::type;
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t w = __builtin_amdgcn_readfirstlane((uint32_t)tid >> 6);
    const uint32_t wm = w >> 1, wn = w & 1u;
    const bool redI32 = I8 && (args.flags & GF_REDUCE_INT32) != 0;
    const bool store = (args.flags & GF_OUTBOUND_STORE) != 0;

    uint32_t *dst = (uint32_t *)(smem + NW * 16384);         // [TABLE] what row i of the tile does
    float *rowScale = (float *)(dst + TABLE);                // [TABLE] W8A8 per-token scale
    // Sums of the tile's tasks (explicit kept rows: of its 128-column halves), [16][half wave]: a place per writer and a fixed
    // order of adding them up, so that sums of floats are the same bits in every launch.
    Sum *sums = (Sum *)(rowScale + TABLE);
    uint32_t *sumTask = (uint32_t *)(sums + 16 * 2 * NW);    // [16]
    __syncthreads();   // every wave has left the main loop's LDS reads behind
    if ((uint32_t)tid < ROWS) {
        const uint32_t v = flex_row<NW == 8>(args, t.row0 + tid);
        uint32_t e = FX_SKIP;
        if ((uint32_t)tid < t.rowsValid) {
            if (v - args.keptBegin < args.keptRows) {   // (unsigned: rows above keptBegin wrap)
                e = FX_KEPT | (v - args.keptBegin);
            } else if (args.flags & GF_ROW_MASK) {
                e = args.checksum ? FX_SUM : FX_SKIP;
            } else if (store || args.checksum) {
                uint32_t ri, task, ws;
                const uint32_t r = fast_div(v, args.fx.dRank, ri);
                flex_task_of(args.sched, r, ri, t.col0 / args.sched.n0, task, ws);
                if (store) {
                    e = FX_OUT | ws;
                } else {   // tiles with checksums hold whole tasks: task g of the tile starts at its row g * mRank
                    const uint32_t g = args.fx.perRank ? 0u : tid / args.sched.mRank;
                    e = FX_SUM | g;
                    sumTask[g] = task;
                }
            }
        }
        dst[tid] = e;
        if constexpr (I8) rowScale[tid] = args.scaleM[flex_row<NW == 8>(args, umin(t.row0 + tid, args.fx.rows - 1u))];
    }
    if (tid < 16 * 2 * NW) sums[tid] = 0;
    __syncthreads();

    unsigned char *st = smem + w * 16384;
    const uint32_t lrow = lane >> 5, chunk = lane & 31;
    const uint32_t lcol = wn * 128u + chunk * 4u;            // the lane's four columns inside the tile
    const bool colOk = lcol < t.colsValid;
    const uint32_t gcol = t.col0 + lcol;
    v4f sN = {1.f, 1.f, 1.f, 1.f};
    v4i bv = {0, 0, 0, 0};
    if constexpr (I8) {
        if (colOk) {
            sN = *(const v4f *)(args.scaleN + gcol);
            if (args.bias) bv = *(const v4i *)(args.bias + gcol);
        }
    }
    // Peers: a base at the tile's first kept row, one 32-bit offset per row from there; a lane with nothing to read gets an
    // offset behind the end of the descriptor (no memory is touched, zeros arrive).  They are fetched for 16 rows of one peer
    // at a time (8 KiB per wave) into a ring of NBUF register buffers that runs on from one 16-row block to the next: while a
    // block adds its last peers the next block's first ones are on their way.  The ring turns a whole number of times per
    // block, with empty descriptors in the turns past the last peer.  (A branch per row instead of
    // selects and out-of-range offsets, and a ring that starts anew for every block: 22.9 instead of 19.8 us at 1024x1024x4096
    // with one peer, bf16, 31.9 instead of 25.3 on 128-row tiles.)
    constexpr int NBUF = 3;
    const uint32_t keptEnd = args.keptBegin + args.keptRows;
    const uint32_t kLo = args.keptBegin > t.row0 ? umin(args.keptBegin - t.row0, t.rowsValid) : 0u;   // the tile's kept rows: [kLo, kLo + kN)
    const bool none = NW == 8 && args.fx.keptInHole != 0;   // (mixed launches)
    const uint32_t kN = !none && keptEnd > t.row0 + kLo ? umin(keptEnd - t.row0, t.rowsValid) - kLo : 0u;
    const int64_t kept0 = (int64_t)t.row0 + kLo - args.keptBegin;   // (of no use, and possibly negative, when the tile has none)
    const bool late = args.fx.late != 0;   // the kept rows' peers are the second launch's
    const bool tileKept = args.nPeers != 0 && kN != 0 && !late;
    const uint32_t peerPitch = (uint32_t)args.peerLd * 4u, lastKept = colOk ? kN : 0u;
    const uint32_t turns = (args.nPeers + NBUF - 1u) / NBUF * NBUF;
    v4i buf[NBUF][8];
    auto fetch = [&](v4i (&b)[8], int blk, uint32_t at) {   // turn `at` of block blk (rows wm*32*MB + 16*blk ..); past its end: of the next
        const bool next = at >= turns;
        const uint32_t p = next ? at - turns : at;
        const float *base = (const float *)args.peers[umin(p, (uint32_t)kMaxRanks - 1u)] + (args.peerRowOffset + kept0) * args.peerLd;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, p < args.nPeers ? 0x7ffffff0 : 0, 0x00020000);
        const uint32_t row = wm * 32 * MB + (blk + (next ? 1 : 0)) * 16 + lrow - kLo;   // (wraps in front of the kept rows)
        const uint32_t end = next && blk + 1 >= 2 * MB ? 0u : lastKept, at0 = row * peerPitch + gcol * 4u;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            b[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, row + 2 * j < end ? at0 + 2 * j * peerPitch : 0xfffffff0u, 0, 2 /* nt */);
    };
    if (tileKept) {
#pragma unroll
        for (int q = 0; q < NBUF - 1; ++q) fetch(buf[q], 0, q);
    }
    // the output the same way: a base at the tile's first kept row, stores of rows that are not kept behind the end
    const uint32_t outPitch = (uint32_t)args.ldd * 2u;
    const __amdgpu_buffer_rsrc_t rd = __builtin_amdgcn_make_buffer_rsrc((void *)((unsigned short *)args.d + kept0 * args.ldd), 0, 0x7ffffff0, 0x00020000);
    Sum run = 0;              // of the rows of task `runOf`, the one this half wave is in (the rows of a task are neighbours)
    uint32_t runOf = (args.flags & GF_ROW_MASK) ? wn : 0u;
    auto flush = [&]() {
        const Sum s = half_sum64(run);
        if (chunk == 31u) sums[runOf * (2u * NW) + w * 2u + lrow] = s;
        run = 0;
    };

#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        flex_stage<L16>(acc, mb, st, lane);
#pragma unroll
        for (int half = 0; half < 2; ++half) {   // 16 rows: a lane has eight of them, two apart
            __builtin_amdgcn_sched_barrier(0);   // (one block's registers at a time)
            v4i cur[8];
            uint32_t d[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t wrow = half * 16 + j * 2 + lrow;
                cur[j] = *(const v4i *)(st + wrow * 512 + ((chunk * 16) ^ flex_turn<L16>(wrow)));
                d[j] = dst[wm * 32 * MB + mb * 32 + wrow];
                if constexpr (I8) cur[j] += bv;
            }
            if (args.accDump) {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint32_t i = wm * 32 * MB + mb * 32 + half * 16 + j * 2 + lrow;
                    if (colOk && i < t.rowsValid) *(v4i *)((int32_t *)args.accDump + (size_t)flex_row<NW == 8>(args, t.row0 + i) * args.N + gcol) = cur[j];
                }
            }
            auto add_peers = [&](auto add) {   // in slot order
                if (!tileKept) return;
                for (uint32_t p = 0; p < turns; p += NBUF) {
#pragma unroll
                    for (int q = 0; q < NBUF; ++q) {
                        __builtin_amdgcn_sched_barrier(0);
                        fetch(buf[(q + NBUF - 1) % NBUF], 2 * mb + half, p + q + NBUF - 1);
                        __builtin_amdgcn_sched_barrier(0);
                        if (p + q < args.nPeers) {
#pragma unroll
                            for (int j = 0; j < 8; ++j) add(cur[j], buf[q][j], j);
                        }
                    }
                }
            };
            const uint32_t blockRow = wm * 32 * MB + mb * 32 + half * 16 + lrow - kLo;   // of row j = 0, counted from the tile's first kept row
            // (32-bit on purpose: the rows in front of the first kept one wrap, and a later row of the same lane is right again)
            auto keptRow = [&](int j) -> uint32_t { return blockRow + 2u * (uint32_t)j; };
            auto isKept = [&](int j) { return keptRow(j) < lastKept; };
            if (late && kN != 0) {   // (wave-uniform)
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (isKept(j)) *(v4i *)(args.skPart + (kept0 + (int64_t)keptRow(j)) * args.N + gcol) = cur[j];
            }
            // (a row that is not kept adds the zeros its loads returned: nothing for int32; floats are added to kept rows only,
            // by selects: a branch per row costs more than the additions)
            if constexpr (I8) {
                if (redI32) add_peers([](v4i &c, const v4i &b, int) { c += b; });
                if (args.cAccum && !late) {
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (isKept(j)) *(v4i *)(args.cAccum + (kept0 + (int64_t)keptRow(j)) * args.N + gcol) = cur[j];
                }
            }
            if (!store && args.checksum) {
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if ((d[j] & FX_KIND) == FX_SUM) {   // (the same for the 32 lanes of a row)
                        const uint32_t g = (args.flags & GF_ROW_MASK) ? wn : (d[j] & FX_INDEX);
                        if (g != runOf) {
                            flush();
                            runOf = g;
                        }
                        Sum v;
                        if constexpr (I8) v = ((long long)cur[j].x + cur[j].y) + ((long long)cur[j].z + cur[j].w);
                        else v = ((double)i2f(cur[j].x) + (double)i2f(cur[j].y)) + ((double)i2f(cur[j].z) + (double)i2f(cur[j].w));
                        run += colOk ? v : (Sum)0;
                    }
            }
            if constexpr (I8) {   // dequantise: per-channel scale first, then per-token, each product rounded on its own
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const bool raw = redI32 && !isKept(j);   // (tiles of other ranks leave as raw int32 there)
                    const float sM = rowScale[wm * 32 * MB + mb * 32 + half * 16 + j * 2 + lrow];
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const int v = f2i(__fmul_rn(__fmul_rn((float)cur[j][c], sN[c]), sM));
                        cur[j][c] = raw ? cur[j][c] : v;
                    }
                }
            }
            if (!redI32)
                add_peers([&](v4i &c, const v4i &b, int j) {
                    const bool k = isKept(j);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int v = f2i(__fadd_rn(i2f(c[e]), i2f(b[e])));
                        c[e] = k ? v : c[e];
                    }
                });
            if (store) {
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (colOk && (d[j] & FX_KIND) == FX_OUT)
                        __builtin_nontemporal_store(cur[j], (v4i *)((float *)args.outbound + (size_t)(d[j] & FX_INDEX) * args.sched.n0 + lcol));
            }
            if (kN != 0 && !late && !(args.flags & GF_KEPT_INT32_ONLY)) {   // (wave-uniform)
                v2i pk[8];
                auto pack = [&](auto cvt) {
#pragma unroll
                    for (int j = 0; j < 8; ++j) {
                        uint32_t q[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) q[e] = cvt(i2f(cur[j][e])) & 0xffffu;
                        pk[j] = v2i{(int)(q[0] | (q[1] << 16)), (int)(q[2] | (q[3] << 16))};
                    }
                };
                if (args.outDtype == DT_BF16) pack([](float f) { return f32_to_bf16_bits(f); });
                else pack([](float f) { return f32_to_f16_bits(f); });
                const uint32_t at0 = blockRow * outPitch + gcol * 2u;
#pragma unroll
                for (int j = 0; j < 8; ++j) __builtin_amdgcn_raw_buffer_store_b64(pk[j], rd, isKept(j) ? at0 + 2 * j * outPitch : 0xfffffff0u, 0, 0);
            }
        }
    }
    if (!store && args.checksum) {
        flush();
        __syncthreads();
        auto total = [&](uint32_t g) {
            Sum s = 0;
            for (uint32_t i = 0; i < 2u * NW; ++i) s += sums[g * (2u * NW) + i];
            return s;
        };
        if (args.flags & GF_ROW_MASK) {
            const uint32_t cols128 = ceil_div(args.N, 128u);
            if (tid < 2 && t.col0 / 128u + tid < cols128) ((Sum *)args.checksum)[(size_t)(t.row0 / 128u) * cols128 + t.col0 / 128u + tid] = total(tid);
        } else {
            // task g of the tile (the only one when row tiles are tile rows of the schedule): its first row says whether it is
            // one of the others', and only then sumTask[g] was written
            const uint32_t g = tid, first = g * args.sched.mRank;
            if (g < (args.fx.perRank ? 1u : 16u) && first < t.rowsValid && (dst[first] & FX_KIND) == FX_SUM) ((Sum *)args.checksum)[sumTask[g]] = total(g);
        }
    }
}

// ---- k slices --------------------------------------------------------------------------------------------------------------
// Few tiles and a long k: every tile's k range is cut into slices, one workgroup each, which store their 32-bit partial sums
// to the workspace as rows of the problem ([slice][row][n]); a second launch adds the slices in slice order and does what
// the epilogue above does.  A second launch costs about what the in-kernel hand-over of the aligned kernels costs (write
// through, count, fetch: a chain of memory round trips on the workgroup that arrives last), and it spreads the rest -- f
// partials and the peers' kept rows, which at few columns outweigh the operands -- over every CU instead of one per tile.
// Explicit kept rows (keptOnly): only they have partial sums in the workspace; what the others add to their checksums is summed
// in registers and leaves as one number per 64 x 128 block and slice.  (With partial sums of all rows and an atomic add per row
// of 128 sums in the second launch 203x1792x4096 with 26 kept rows took 22.0 us instead of 13.7, 128x1024x8192 with 16 27.1
// instead of 12.6.)
// The same second launch also serves whole tiles whose kept rows leave as sums (late): it then adds nothing but their peers.
template <int MB, typename Acc>
__device__ __forceinline__ void flex_store_partial(const GemmArgs &args, Acc (&acc)[MB][4], unsigned char *smem, const FlexTile &t, uint32_t slice)
{
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t w = __builtin_amdgcn_readfirstlane((uint32_t)tid >> 6);
    const uint32_t wm = w >> 1, wn = w & 1u;
    const int c32 = lane & 31, h = lane >> 5;
    uint32_t kLo = 0, kHi = t.rowsValid;   // the tile's rows whose partial sums are stored
    if constexpr (std::is_same<Acc, v16i>::value) {
        if (args.fx.keptOnly) {
            const uint32_t end = t.row0 + t.rowsValid;
            kLo = args.keptBegin > t.row0 ? umin(args.keptBegin - t.row0, t.rowsValid) : 0u;
            kHi = umin(args.keptBegin + args.keptRows, end) - umin(t.row0, umin(args.keptBegin + args.keptRows, end));
            if (args.checksum) {   // the other rows leave as one sum per 64 x 128 block
                const uint32_t col = wn * 128u + c32, cols128 = ceil_div(args.N, 128u), c = t.col0 / 128u + wn;
                long long sum = 0;
                uint32_t others = 0;   // rows of this lane that are not kept
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const uint32_t row = wm * 32 * MB + mb * 32 + (r >> 2) * 8 + h * 4 + (r & 3);
                        const bool other = row < t.rowsValid && !(row >= kLo && row < kHi);
                        others += other ? 1u : 0u;
#pragma unroll
                        for (int nb = 0; nb < 4; ++nb) sum += other && col + nb * 32 < t.colsValid ? (long long)acc[mb][nb][r] : 0ll;
                    }
                if (slice == 0 && args.bias) {
#pragma unroll
                    for (int nb = 0; nb < 4; ++nb)
                        if (col + nb * 32 < t.colsValid) sum += (long long)args.bias[t.col0 + col + nb * 32] * others;
                }
                sum = wave_sum64(sum);
                long long *sums = (long long *)(smem + FLEX_STAGING);
                __syncthreads();   // (every wave has left the main loop's LDS reads behind)
                if (lane == 63) sums[w] = sum;
                __syncthreads();
                if (wm == 0 && lane == 0 && c < cols128) {
                    long long *to = args.fx.sliceSums + ((size_t)(t.row0 / 128u) * cols128 + c) * 2u * args.fx.slices + 2u * slice;
                    to[(t.row0 / 64u) & 1u] = sums[wn] + sums[2 + wn];
                }
            }
            if (kLo >= kHi) return;
        }
    }
    // checksums of whole numbers: the second launch adds to them (sums of floats are added up by a third, in row order)
    if (std::is_same<Acc, v16i>::value && !args.fx.keptOnly && slice == 0 && args.checksum != nullptr && !(args.flags & GF_OUTBOUND_STORE) && (uint32_t)tid < t.rowsValid) {
        const uint32_t v = t.row0 + tid;
        long long *sum = (long long *)args.checksum;
        if (args.flags & GF_ROW_MASK) {
            const uint32_t cols128 = ceil_div(args.N, 128u), c = t.col0 / 128u;
            sum[(size_t)(v / 128u) * cols128 + c] = 0;
            if (c + 1u < cols128) sum[(size_t)(v / 128u) * cols128 + c + 1u] = 0;
        } else if (v - args.keptBegin >= args.keptRows) {
            uint32_t ri, task, ws;
            const uint32_t r = fast_div(v, args.fx.dRank, ri);
            flex_task_of(args.sched, r, ri, t.col0 / args.sched.n0, task, ws);
            sum[task] = 0;
        }
    }
    __syncthreads();   // every wave has left the main loop's LDS reads behind
    unsigned char *st = smem + w * 16384;
    const uint32_t lrow = lane >> 5, chunk = lane & 31, lcol = wn * 128u + chunk * 4u;
    // (signed: the tile's first row may lie in front of the kept ones, which alone are stored)
    const int64_t row0 = args.fx.keptOnly ? (int64_t)slice * args.keptRows + t.row0 - args.keptBegin : (int64_t)slice * args.fx.rows + t.row0;
    int32_t *part = args.skPart + row0 * args.N + t.col0 + lcol;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        if (wm * 32 * MB + mb * 32 >= kHi || wm * 32 * MB + mb * 32 + 32 <= kLo) continue;   // (wave-uniform)
        flex_stage<false>(acc, mb, st, lane);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const uint32_t wrow = j * 2 + lrow, i = wm * 32 * MB + mb * 32 + wrow;
            const v4i v = *(const v4i *)(st + wrow * 512 + ((chunk * 16) ^ flex_turn<false>(wrow)));
            if (i >= kLo && i < kHi && lcol < t.colsValid) *(v4i *)(part + (size_t)i * args.N) = v;
        }
    }
}

// Workgroup (ct, y): columns [256 ct, +256) of rows [rowsPer * y, +rowsPer).  A wave takes one row at a time (everything about
// the row is wave-uniform), a lane four columns of it: partials and peers are 1 KiB per wave instruction, all of them
// requested before the first is used.
template <uint32_t DT>
__global__ void __launch_bounds__(256) flex_finish_kernel(const GemmArgs args, const uint32_t rowsPer)
{
    constexpr bool I8 = DT == DT_I8;
    using Sum = typename std::conditional<I8, unsigned long long, double>::type;
    // (named here, the arguments arrive in a few wide loads: they come from host memory)
    const void *peer[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) peer[q] = args.peers[q];
    asm volatile("" : : "s"(peer[0]), "s"(peer[1]), "s"(peer[2]), "s"(peer[3]), "s"(peer[4]), "s"(peer[5]), "s"(peer[6]), "s"(peer[7]), "s"(args.skPart), "s"(args.d),
                 "s"(args.scaleM), "s"(args.scaleN), "s"(args.bias), "s"(args.checksum), "s"(args.accDump), "s"(args.cAccum), "s"(args.ldd), "s"(args.peerLd), "s"(args.peerRowOffset),
                 "s"(args.N), "s"(args.flags), "s"(args.nPeers), "s"(args.keptBegin), "s"(args.keptRows), "s"(args.outDtype), "s"(args.fx.slices), "s"(args.fx.sliceSums));
    const int lane = threadIdx.x & 63;
    const uint32_t w = __builtin_amdgcn_readfirstlane((uint32_t)threadIdx.x >> 6);
    const bool redI32 = I8 && (args.flags & GF_REDUCE_INT32) != 0;
    const bool store = (args.flags & GF_OUTBOUND_STORE) != 0, rowMask = (args.flags & GF_ROW_MASK) != 0;
    const bool sums = !store && args.checksum != nullptr;
    const bool keptOnly = I8 && args.fx.keptOnly != 0, late = args.fx.late != 0;
    const uint32_t first = keptOnly || late ? args.keptBegin : 0u, stored = keptOnly || late ? args.keptRows : args.fx.rows;   // the rows the partial sums hold
    const uint32_t row0 = first + blockIdx.y * rowsPer, rowEnd = umin(row0 + rowsPer, first + stored);
    const uint32_t lcol = lane * 4u, gcol = blockIdx.x * 256u + lcol;
    const bool colOk = gcol < args.N;
    const uint32_t slices = args.fx.slices;
    v4f sN = {1.f, 1.f, 1.f, 1.f};
    v4i bv = {0, 0, 0, 0};
    if constexpr (I8) {
        if (colOk) {
            sN = *(const v4f *)(args.scaleN + gcol);
            if (args.bias) bv = *(const v4i *)(args.bias + gcol);
        }
    }
    if constexpr (I8) {
        if (keptOnly && args.checksum) {   // a wave per 128 x 128 block of this column tile
            const uint32_t cols128 = ceil_div(args.N, 128u), blocks = ceil_div(args.fx.rows, 128u) * 2u;
            for (uint32_t e = blockIdx.y * 4u + (w ^ 3u); e < blocks; e += gridDim.y * 4u) {   // (few rows: they are the first waves')
                const uint32_t rb = e >> 1, c = blockIdx.x * 2u + (e & 1u);
                if (c >= cols128) continue;
                const long long *from = args.fx.sliceSums + ((size_t)rb * cols128 + c) * 2u * slices;
                const bool both = rb * 128u + 64u < args.fx.rows;   // (the last block may have no lower half)
                long long s = 0;
                for (uint32_t i = lane; i < 2u * slices; i += 64u)
                    if (both || (i & 1u) == 0) s += from[i];
                s = wave_sum64(s);
                if (lane == 63) ((long long *)args.checksum)[(size_t)rb * cols128 + c] = s;
            }
        }
    }
    // Checksums of whole numbers: a task's rows add to one address, one atomic after the other (0.15 us each), so the waves of a
    // workgroup meet in LDS first (504x4112x1024, eight ranks, an atomic per row / per workgroup: 32.3 / 24.5 us).  Floats
    // are not added in order of arrival: a row's sum takes the place of the row's partial sums, which nobody reads again, for
    // flex_sums_kernel.
    __shared__ Sum waveSum[4];
    __shared__ uint32_t waveTask[4];
    Sum run = 0;
    uint32_t runOf = 0xffffffffu;
    // A row's addresses are wave-uniform but for the lane's columns: descriptors in scalar registers and one offset register for
    // every load.  (With 64-bit addresses in vector registers the compiler at times puts them where an earlier load is still to
    // arrive, and waits for it: the peers' loads then go one by one, bf16 all-reduce 16x8192x1024 of eight ranks 13.0 / 13.8 us.)
    const uint32_t laneAt = lane * 16u;
    auto load = [&](const int32_t *p, auto aux) {
        return __builtin_amdgcn_raw_buffer_load_b128(__builtin_amdgcn_make_buffer_rsrc((void *)p, 0, 1024, 0x00020000), laneAt, 0, decltype(aux)::value);
    };
    constexpr std::integral_constant<int, 0> KEEP{};
    constexpr std::integral_constant<int, 2> NT{};
    for (uint32_t v = row0 + w; v < rowEnd; v += 4u) {
        const bool kept = v - args.keptBegin < args.keptRows;
        // the peers first: they do not wait for the sums
        const uint32_t nP = kept ? args.nPeers : 0u;
        const size_t peerAt = kept ? (size_t)(args.peerRowOffset + (v - args.keptBegin)) * args.peerLd + blockIdx.x * 256u : 0;
        v4i pv[8], cur = {0, 0, 0, 0};
        if (colOk) {
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if ((uint32_t)q < nP) pv[q] = load((const int *)peer[q] + peerAt, NT);
            const int32_t *part = args.skPart + (size_t)(v - first) * args.N + blockIdx.x * 256u;
            const size_t pitch = (size_t)stored * args.N;
            auto add_part = [&](const v4i &t) {
                if constexpr (I8) {
                    cur += t;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) cur[e] = f2i(__fadd_rn(i2f(cur[e]), i2f(t[e])));
                }
            };
            uint32_t s0 = 0;   // (whole eights without a branch per slice: with the arguments named above, bf16 all-reduce 2x12800x576 in 34 slices 14.0 -> 13.0 us)
            for (; s0 + 8u <= slices; s0 += 8u) {
                v4i t[8];
#pragma unroll
                for (int q = 0; q < 8; ++q) t[q] = load(part + (s0 + q) * pitch, KEEP);
#pragma unroll
                for (int q = 0; q < 8; ++q) add_part(t[q]);
            }
            v4i t[7];
#pragma unroll
            for (int q = 0; q < 7; ++q)
                if (s0 + q < slices) t[q] = load(part + (s0 + q) * pitch, KEEP);
#pragma unroll
            for (int q = 0; q < 7; ++q)
                if (s0 + q < slices) add_part(t[q]);
            if (I8 && !late) cur += bv;   // (late: the first launch has added the bias and written the dump)
            if (args.accDump && !late) *(v4i *)((int32_t *)args.accDump + (size_t)v * args.N + gcol) = cur;
        }
        if (!kept) {
            uint32_t ws = 0, task = 0;
            if (!rowMask) {
                uint32_t ri;
                const uint32_t r = fast_div(v, args.fx.dRank, ri);
                flex_task_of(args.sched, r, ri, blockIdx.x * 256u / args.sched.n0, task, ws);
            }
            if (sums) {
                Sum s = 0;
                if (colOk) {
                    if constexpr (I8) s = (Sum)(((long long)cur.x + cur.y) + ((long long)cur.z + cur.w));
                    else s = ((double)i2f(cur.x) + (double)i2f(cur.y)) + ((double)i2f(cur.z) + (double)i2f(cur.w));
                }
#pragma unroll
                for (int o = 16; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
                if constexpr (I8) {
                    Sum *to = (Sum *)args.checksum;
                    if (rowMask) {   // one sum per 128 columns
                        if ((lane & 31) == 0 && colOk) atomicAdd(to + (size_t)(v / 128u) * ceil_div(args.N, 128u) + gcol / 128u, s);
                    } else {
                        s += __shfl_xor(s, 32, 64);
                        if (task != runOf) {
                            if (lane == 0 && runOf != 0xffffffffu) atomicAdd(to + runOf, run);
                            run = 0;
                            runOf = task;
                        }
                        run += s;
                    }
                } else {
                    s += __shfl_xor(s, 32, 64);
                    if (lane == 0) *(double *)(args.skPart + (size_t)(v - first) * args.N + gcol) = s;   // (8 bytes of at least 16)
                }
            }
            if (store && colOk) {
                if constexpr (I8) {
                    if (!redI32) {
                        const float sM = args.scaleM[v];
#pragma unroll
                        for (int e = 0; e < 4; ++e) cur[e] = f2i(__fmul_rn(__fmul_rn((float)cur[e], sN[e]), sM));
                    }
                }
                __builtin_nontemporal_store(cur, (v4i *)((float *)args.outbound + (size_t)ws * args.sched.n0 + lcol));
            }
            continue;
        }
        if (!colOk) continue;
        auto addPeers = [&](auto add) {
            for (uint32_t p0 = 0; p0 < nP; p0 += 8u) {
                if (p0) {
#pragma unroll
                    for (int q = 0; q < 8; ++q)
                        if (p0 + q < nP) pv[q] = load((const int *)args.peers[p0 + q] + peerAt, NT);
                }
#pragma unroll
                for (int q = 0; q < 8; ++q)
                    if (p0 + q < nP) add(pv[q]);
            }
        };
        if constexpr (I8) {
            if (redI32) addPeers([&](const v4i &b) { cur += b; });
            if (args.cAccum) *(v4i *)(args.cAccum + (size_t)(v - args.keptBegin) * args.N + gcol) = cur;
            const float sM = args.scaleM[v];
#pragma unroll
            for (int e = 0; e < 4; ++e) cur[e] = f2i(__fmul_rn(__fmul_rn((float)cur[e], sN[e]), sM));
        }
        if (!redI32)
            addPeers([&](const v4i &b) {
#pragma unroll
                for (int e = 0; e < 4; ++e) cur[e] = f2i(__fadd_rn(i2f(cur[e]), i2f(b[e])));
            });
        uint32_t q[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) q[e] = f32_to_out16(i2f(cur[e]), args.outDtype) & 0xffffu;
        *(v2i *)((unsigned short *)args.d + (size_t)(v - args.keptBegin) * args.ldd + gcol) = v2i{(int)(q[0] | (q[1] << 16)), (int)(q[2] | (q[3] << 16))};
    }
    if (I8 && sums && !rowMask) {
        if (lane == 0) {
            waveSum[w] = run;
            waveTask[w] = runOf;
        }
        __syncthreads();
        if (threadIdx.x < 4u) {   // the first wave of a task adds for all of them
            const uint32_t mine = waveTask[threadIdx.x];
            Sum all = 0;
            bool firstOf = mine != 0xffffffffu;
            for (uint32_t i = 0; i < 4u; ++i)
                if (waveTask[i] == mine) {
                    if (i < threadIdx.x) firstOf = false;
                    all += waveSum[i];
                }
            if constexpr (I8) {
                if (firstOf) atomicAdd((Sum *)args.checksum + mine, all);
            }
        }
    }
}

// Checksums of float launches in k slices: workgroup b * colTiles + ct, one wave, is the task of column tile ct in tile row b of
// all ranks' tile rows, and adds the sums of its rows (at most 128) that flex_finish_kernel left in slice 0, always in the same
// order.
// A launch more than adding in order of arrival in flex_finish_kernel, whose last bits differ from launch to launch; bf16, eight
// ranks, us: 504x4112x1024 21.1 / 22.1, 88x1024x4096 13.6 / 14.8, 64x4096x8192 22.5 / 24.2.
template <uint32_t DT>
__global__ void __launch_bounds__(64) flex_sums_kernel(const GemmArgs args)
{
    const SchedParams &sp = args.sched;
    const uint32_t b = blockIdx.x / args.fx.colTiles, ct = blockIdx.x - b * args.fx.colTiles, rank = b / sp.loopsM, mi = b - rank * sp.loopsM;
    const uint32_t row0 = rank * sp.mRank + mi * sp.m0, rows = umin(sp.m0, sp.mRank - mi * sp.m0);
    if (row0 - args.keptBegin < args.keptRows) return;
    const int32_t *from = args.skPart + (size_t)row0 * args.N + ct * 256u;
    double s = 0;
    for (uint32_t r = threadIdx.x; r < rows; r += 64u) s += *(const double *)(from + (size_t)r * args.N);
    uint32_t task, ws;
    flex_task_of(sp, rank, mi * sp.m0, ct, task, ws);
    s = wave_sum64(s);
    if (threadIdx.x == 63) ((double *)args.checksum)[task] = s;
}

}  // namespace catcoc
