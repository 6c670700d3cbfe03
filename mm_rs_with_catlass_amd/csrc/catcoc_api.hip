// C ABI of libcatcoc_hip.so: argument validation, tiling selection and dispatch
// to the fused GEMM kernels.  Declarations and the reference interfaces they
// replace are in include/catcoc_hip.h.
#include <hip/hip_runtime.h>
#include <pthread.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <math.h>

#include <new>
#include <vector>

#include "catcoc_hip.h"
#include "comm_reduce.h"
#include "gemm_args.h"
#include "tile_sched.h"

namespace catcoc {
int launch_gemm_i8(const GemmArgs &args, int variant, bool edge, void *stream);
int launch_gemm_dma_i8(const GemmArgs &args, void *stream);
int launch_gemm_splitk_i8(const GemmArgs &args, int rowBlocks, uint32_t tasks, void *stream);
int launch_gemm_decode_nk_i8(const GemmArgs &args, void *stream);
int launch_gemm_f16(const GemmArgs &args, int variant, bool edge, void *stream);
int launch_gemm_bf16(const GemmArgs &args, int variant, bool edge, void *stream);
int launch_gemm_dma_f16(const GemmArgs &args, void *stream);
int launch_gemm_dma_bf16(const GemmArgs &args, void *stream);
int launch_gemm_flex_i8(const GemmArgs &args, int rowBlocks, void *stream);
int launch_gemm_flex_f16(const GemmArgs &args, int rowBlocks, void *stream);
int launch_gemm_flex_bf16(const GemmArgs &args, int rowBlocks, void *stream);
int launch_gemm_mid(uint32_t dtype, const GemmArgs &args, int tileRows, void *stream);
int launch_gemm_mixed(uint32_t dtype, const GemmArgs &args, void *stream);
int launch_gemm_few(uint32_t dtype, const GemmArgs &args, int tileRows, int tileCols, void *stream);

// What the calling thread launched last (catcoc_last_launch).
static thread_local CatcocLaunchInfo g_launch;

static int launch_flex(uint32_t dtype, const GemmArgs &args, int rowBlocks, void *stream)
{
    g_launch = {CATCOC_KERNEL_FLEXIBLE, 64u * rowBlocks, 256, args.fx.slices > 1 ? args.fx.slices : 1u, 0, 0};
    switch (dtype) {
        case DT_I8: return launch_gemm_flex_i8(args, rowBlocks, stream);
        case DT_F16: return launch_gemm_flex_f16(args, rowBlocks, stream);
        case DT_BF16: return launch_gemm_flex_bf16(args, rowBlocks, stream);
        default: return (int)hipErrorInvalidValue;
    }
}

static int launch_gemm(uint32_t dtype, const GemmArgs &args, int variant, bool edge, void *stream)
{
    g_launch = {CATCOC_KERNEL_GENERAL, args.sched.m0, args.sched.n0, 1, 0, 0};
    switch (dtype) {
        case DT_I8: return launch_gemm_i8(args, variant, edge, stream);
        case DT_F16: return launch_gemm_f16(args, variant, edge, stream);
        case DT_BF16: return launch_gemm_bf16(args, variant, edge, stream);
        default: return (int)hipErrorInvalidValue;
    }
}

static int launch_gemm_dma(uint32_t dtype, const GemmArgs &args, void *stream)
{
    g_launch = {CATCOC_KERNEL_ALIGNED, args.sched.m0, args.sched.n0, args.splitK > 1 ? args.splitK : 1u, 0, 0};
    switch (dtype) {
        case DT_I8: return launch_gemm_dma_i8(args, stream);
        case DT_F16: return launch_gemm_dma_f16(args, stream);
        case DT_BF16: return launch_gemm_dma_bf16(args, stream);
        default: return (int)hipErrorInvalidValue;
    }
}
}

using namespace catcoc;

namespace {

thread_local char g_err[512] = "";
thread_local int g_status = 0;

int fail(int code, const char *fmt, ...)
{
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    g_status = code;
    return code;
}

void ok()
{
    g_err[0] = 0;
    g_status = 0;
}

enum { E_NULL = 1, E_DESC = 2, E_SHAPE = 3, E_RANK = 4, E_TILING = 5, E_DTYPE = 6, E_WORKSPACE = 7, E_LAUNCH = 8 };

void launched(int e)
{
    if (e) fail(E_LAUNCH, "kernel launch failed: %s", hipGetErrorString((hipError_t)e));
    else ok();
}

constexpr uint32_t kDefaultBlockNum = 256;  // one scheduling slot per CU of an MI355X
constexpr uint32_t kDefaultStages = 2;      // WORKSPACE_STAGES, examples/dynamic_tiling/include/info.h:18
// Every workspace starts with one block of per-tile arrival counters at a fixed place and of a fixed size, whatever the
// shape or slice count of the launch: launches of different shapes can then share one workspace that was zeroed once
// (each launch leaves its counters at zero again; the partial tiles behind the block are written before they are read).
constexpr uint64_t kCounterBlockBytes = CATCOC_WORKSPACE_COUNTER_BYTES;
constexpr uint32_t kMaxCountedTiles = (uint32_t)(kCounterBlockBytes / 4u);

struct Plan {
    GemmArgs args;
    int variant;  // 0 = general kernel, else tile rows / 64 of the fast kernel
    bool edge;
    uint32_t dtype;
    uint32_t blockNum;
    bool dma;     // full tiles, row-major operands: the direct-to-LDS kernel applies
    bool preferFlex;         // run there although the aligned kernels would take it
    uint32_t *counters;      // the workspace's counter block (NULL: none), and the bytes behind it that the launch may use
    uint64_t room;
    bool maySmall;           // the caller left tiles, slices and order to the library: small tiles are a choice (small_tile)
    int flexBlocks;          // 0 = no; else the launch can run in flexible mode (gemm_flex.h) on tiles of 64 * flexBlocks rows
    uint32_t kSlices;        // k slices per tile this launch would run with a workspace (1 = none)
    uint64_t kSliceBytes;    // workspace for that: partial tiles + counters
};

uint32_t elem_size(uint32_t dt) { return dt == DT_I8 ? 1u : 2u; }

// Flexible mode (gemm_flex.h) for a launch whose schedule, kept rows and flags are filled in: fills args.fx and returns the
// tile's rows / 64, or 0 when the launch cannot run there (A as [k,m], rows of k not in 4-byte pieces, n no multiple of
// four, tiles of another width).  `sums` = checksums were asked for and the tiles run whole: a row tile then holds whole tasks.  wantM0 =
// the caller's tile rows (0: the library's choice), slices = k slices per tile.
int plan_flex(GemmArgs &a, uint32_t es, bool sums, uint32_t wantM0, uint32_t slices)
{
    const SchedParams &s = a.sched;
    const uint64_t kBytes = (uint64_t)a.K * es;
    if (a.transA || s.n0 != 256 || (s.m0 != 64 && s.m0 != 128) || kBytes % 4 != 0 || a.N % 4 != 0 || kBytes > 0x7fffffffull) return 0;
    FlexParams &f = a.fx;
    const uint64_t rows = s.op == OP_ALLGATHER ? (uint64_t)a.M * s.P : a.M;
    if (rows >= (1u << 30)) return 0;
    f.rows = (uint32_t)rows;
    f.colTiles = ceil_div(a.N, 256u);
    f.slices = slices;
    f.late = 0;
    f.dRank = make_fast_div(s.mRank);
    // the step of k that goes through registers with bounds checks: what whole steps leave, and the last step of all when
    // rows of B end inside a 16-byte piece (the copies then read past the end of every row but the last)
    f.tail = (uint32_t)(kBytes % 64);
    if (f.tail == 0 && !a.transB && ((uint64_t)a.N * es) % 16 != 0) f.tail = 64;
    // 64-row tiles as long as they are at most one per CU (measured figures: make_plan)
    int blocks = wantM0 ? (int)(wantM0 / 64u) : slices > 1 || ceil_div(f.rows, 64u) * f.colTiles <= 256u ? 1 : 2;
    f.perRank = 0;
    f.rowStep = 64u * blocks;
    if (sums && slices <= 1) {
        if (a.flags & GF_ROW_MASK) {                 // checksums per 128 x 128 block
            if (f.rows > 64u) blocks = 2;
            f.rowStep = 64u * blocks;
        } else if (s.op == OP_REDUCE_SCATTER && s.P > 1) {
            if (s.loopsM > 1) {                      // a task is one tile row of one rank
                f.perRank = 1;
                blocks = (int)(s.m0 / 64u);
            } else {                                 // a task is a rank's rows (at most m0)
                if (s.mRank > 64u) blocks = 2;
                f.rowStep = 64u * blocks / s.mRank * s.mRank;
            }
        }
    }
    f.rowTiles = f.perRank ? s.P * s.loopsM : ceil_div(f.rows, f.rowStep);
    f.keptTile0 = 0;
    f.keptTiles = 0;
    if (s.op == OP_REDUCE_SCATTER && s.P > 1) {
        f.keptTile0 = f.perRank ? a.keptRank * s.loopsM : a.keptBegin / f.rowStep;
        f.keptTiles = f.perRank ? s.loopsM : (a.keptBegin + a.keptRows - 1u) / f.rowStep + 1u - f.keptTile0;
    }
    return blocks;
}

// k slices per tile a launch in flexible mode takes by itself.  A workgroup's k step takes 0.3 us as long as the CUs are not
// full; a slice costs the second launch about 0.1 us of latency and rows x n words written and read back at 4 TB/s.  The sum
// steps * 0.3 / f + f * (0.1 + 2e-6 * rows * n) is least at the root below.  Measured optimum / this rule, bf16 all-reduce:
// 16x8192x1024 24 / 24, 100x8192x1024 16 / 16, 28x15360x768 32 / 31, 16x4096x4096 8-16 / 13, 64x2048x4096 6 / 6,
// 100x1024x8192 2 / 2, 200x1024x2048 3 / 3, 400x6144x1024 8 / 8, 824x7296x1280 3 / 3.
// At most one workgroup per CU, except where that leaves a fifth of the CUs idle (or, for 16-bit operands, allows two slices
// only) and k is long: then two per CU, if the root asks for as many.  One -> two, bf16 all-reduce, one peer, B as [n,k] / [k,n],
// us: 88 tiles, 512 steps 149 / 139 -> 87 / 76; 98 tiles, 484 steps 167 / 124 -> 102 / 87; 128 tiles, 256 steps 76 / 68 -> 63 / 56;
// 160 tiles, 512 steps 379 / 221 -> 258 / 153.  Not where the CUs are busy: W8A8, 120 tiles, 255 steps 82 / 55 -> 92 / 62;
// bf16, 64 tiles, 512 steps 78 / 66 -> 79 / 71, 240 tiles, 384 steps 219 / 127 -> 286 / 163.
uint32_t flex_slices(uint32_t es, uint32_t rows, uint32_t n, uint32_t tiles, uint32_t steps)
{
    const double f = sqrt(0.3 * steps / (0.1 + 2e-6 * (double)rows * (double)n));
    const uint32_t least = umin((uint32_t)(f + 0.5), umin(steps / 4u, 64u)), once = tiles ? 256u / tiles : 1u, twice = tiles ? 512u / tiles : 1u;
    const bool pays = steps >= 256u && least >= twice && once <= 2u && (tiles * once <= 200u || (es == 2u && once == 2u));
    const uint32_t r = pays ? twice : umin(least, once);
    return r < 2u ? 1u : r;
}

// Reduce-scatter launches of one round of tiles: the few workgroups with kept rows stream all the peers (64 KiB per peer and 64
// rows, at about 35 GB/s per CU) while the other CUs are done.  With the workspace the query asks for, the kept rows leave as
// 32-bit sums and a second launch adds the peers over every CU.  One launch / two, us, launches alternating: W8A8 P = 8
// 1000x1376x4096 27.3 / 25.5 (checksums 32.6 / 25.9), 504x1376x4096 21.7 / 19.3, 4000x1376x2048 42.3 / 34.4, 1016x736x1024
// 17.8 / 16.2; bf16 P = 8 800x1040x4096 25.4 / 22.3, 2000x1040x4096 41.9 / 32.9.  Below 256 KiB of peers per tile the second launch
// (2-3 us) has nothing to win (bf16 P = 4 200x1040x8192, 150 KiB: 18.0 / 20.4 us; not taken).
bool flex_late(const GemmArgs &a)
{
    const SchedParams &s = a.sched;
    return s.op == OP_REDUCE_SCATTER && s.P > 1 && !(a.flags & (GF_ROW_MASK | GF_KEPT_INT32_ONLY)) && a.fx.rowTiles * a.fx.colTiles <= 256u &&
           a.nPeers * umin(a.keptRows, 64u) >= 256u;
}

// Tiles and k slices of a launch that may run in flexible mode, in two halves: what it would take, and what it takes of the
// workspace it is given.  A launch is given no more of its workspace than its query asks for (the rest may be another
// launch's), so the first half must not depend on the operands' layouts, which the query does not know.
struct FlexSlices {
    int whole;             // rows / 64 of its tiles without k slices; 0: it cannot run in flexible mode
    uint32_t slices;       // k slices with a large enough workspace
    uint64_t bytes;        // what they take (one slice and some bytes: the peers' second launch)
    uint64_t slice, sums;  // of that per slice: all, and the sums of rows that are not kept
    bool keptOnly;
};

// Fills args.fx for whole tiles.  wantSlices = the caller's own number (0: the library's).
FlexSlices flex_choose(GemmArgs &a, uint32_t es, uint32_t wantM0, uint32_t wantSlices)
{
    const bool sums = (a.flags & GF_OUTBOUND_STORE) == 0 && a.checksum != nullptr;
    FlexSlices c = {plan_flex(a, es, sums, wantM0, 1), 1, 0, 0, 0, false};
    if (c.whole == 0) return c;
    // (whole k steps as with B as [k,n]: with B as [n,k] there is one more where rows of B would end inside a 16-byte piece)
    const uint64_t kBytes = (uint64_t)a.K * es;
    const uint32_t steps = (uint32_t)(kBytes / 64u) - (kBytes % 64u == 0 && ((uint64_t)a.N * es) % 16u != 0 ? 1u : 0u);
    const uint32_t tiles = ceil_div(a.fx.rows, 64u) * a.fx.colTiles;
    // explicit kept rows: the other rows need no partial sums of their own (the dump, if there is one, does)
    c.keptOnly = (a.flags & GF_ROW_MASK) != 0 && a.accDump == nullptr;
    const uint32_t stored = c.keptOnly ? a.keptRows : a.fx.rows;
    uint32_t own = flex_slices(es, stored, a.N, tiles, steps);
    // (a reduce-scatter's other rows are done after the first launch: two slices' traffic is more than they save.  Whole / two
    // slices, bf16, four ranks, 200x1040x8192 18.1 / 33.2 with checksums, 18.8 / 23.6 us with stored tiles)
    if (own == 2 && !c.keptOnly && a.sched.op == OP_REDUCE_SCATTER && a.sched.P > 1) own = 1;
    const uint32_t f = umin(umin(wantSlices ? wantSlices : own, 64u), steps);
    if (f <= 1) {
        if (wantSlices <= 1 && flex_late(a)) c.bytes = kCounterBlockBytes + (uint64_t)a.keptRows * a.N * 4u;
        return c;
    }
    c.slices = f;
    c.sums = c.keptOnly && sums ? (uint64_t)ceil_div(a.fx.rows, 128u) * ceil_div(a.N, 128u) * 16u : 0u;
    c.slice = ((uint64_t)stored * a.N * 4u + c.sums + 15u) / 16u * 16u;
    c.bytes = kCounterBlockBytes + f * c.slice;
    return c;
}

// The slices that fit (none: whole tiles), in args.fx; returns the tile's rows / 64.
int flex_use(GemmArgs &a, uint32_t es, uint32_t wantM0, const FlexSlices &c, void *workspace, uint64_t workspaceBytes)
{
    if (c.bytes == 0 || workspace == nullptr || (uintptr_t)workspace % 256 != 0) return c.whole;
    unsigned char *part = (unsigned char *)workspace + kCounterBlockBytes;
    if (c.slices <= 1) {
        if (workspaceBytes >= c.bytes) {
            a.fx.late = 1;
            a.skPart = (int32_t *)part;
        }
        return c.whole;
    }
    if (workspaceBytes < kCounterBlockBytes + 2u * c.slice) return c.whole;
    const uint64_t fit = (workspaceBytes - kCounterBlockBytes) / c.slice;
    const uint32_t run = fit < c.slices ? (uint32_t)fit : c.slices;
    a.fx.keptOnly = c.keptOnly ? 1u : 0u;
    a.fx.sliceSums = (long long *)part;
    a.skPart = (int32_t *)(part + run * c.sums);
    return plan_flex(a, es, (a.flags & GF_OUTBOUND_STORE) == 0 && a.checksum != nullptr, wantM0, run);
}

// What flexible mode asks of the pointers: operands on the 4-byte grid, everything the epilogue touches in its 8- and 16-byte
// accesses on theirs.
bool flex_ptrs_ok(const GemmArgs &a)
{
    auto on = [](const void *p, uintptr_t g) { return (uintptr_t)p % g == 0; };
    if (!on(a.b, 4) || !on(a.d, 8) || !on(a.scaleN, 16) || !on(a.bias, 16) || !on(a.cAccum, 16) || !on(a.accDump, 16) || !on(a.outbound, 16)) return false;
    for (uint32_t r = 0; r < a.sched.P || r == 0; ++r)
        if (!on(a.a[r], 4)) return false;
    // (the epilogue addresses the peers' and the output's rows of a tile with 31-bit offsets from the tile's first one)
    if ((a.nPeers && (a.peerLd % 4 != 0 || (uint64_t)a.peerLd * 4u * 160u > 0x7fffffffull)) || (uint64_t)a.ldd * 2u * 160u > 0x7fffffffull) return false;
    for (uint32_t p = 0; p < a.nPeers; ++p)
        if (!on(a.peers[p], 16)) return false;
    return true;
}

// ---- one launch of small or mixed tiles (gemm_few.h, gemm_mid.h, gemm_mixed.h) or the other kernels ------------------------------------
// Both sides of the choice are estimates in us, fitted to 460 calls of every operator (1 to 8192 rows, k 512 to 16384, n 512 to 8192,
// 2 to 8 ranks, up to 6e11 operations, GPU time of calls behind each other; what concerns slices, sums, dealt rows and whole rounds of
// few tiles, to another 480): what a launch costs by itself, per round of workgroups (128 columns: per workgroup of a CU), per
// KiB a workgroup pulls in through its CU (more from the second round of workgroups on: the first leaves the caches cold), per MB of
// operands, per MB of peers and outputs; rows of k off the 16-byte grid and B as [k,n] cost more per KiB, rows of a B tile that are no whole
// cache line more per MB.  Half of the estimates are within 0.10 of the tiles' times and 0.06 of the others', nine in ten within 0.22
// and 0.16.  The tiles of 96, 160 and 192 rows stand on the scale of the 128-row one's (their times relative to it, 1600 calls).  The estimates of
// 128-column tiles are from when these ran 32x32 MFMAs and come out up to 0.2 high, of flexible tiles in k slices 0.12, so the choice, the tiles with the least, compares
// shares (other_share), set on 7100 drawn calls, each timed on every tile in reach.  2100 others take 0.913 of the time they took before
// the 16x16 MFMAs and the tiles of 96, 160 and 192 rows, 25 of them more than 1.04; with the shares and the estimate of mixed launches that those came with 0.923, 61 of them.
// For calls unlike those (k below 512, columns that are no multiple of 32, one rank or more than eight) the shares are older and the tiles of 96, 160 and 192 rows
// left out: 283 drawn ones take 1.032 of the best choice's time, and none lost more than 0.04 by the re-fitted estimates of mixed launches.
// Figures of calls stand with the kernels that run them (gemm_few.h, gemm_mid.h, gemm_mixed.h).
constexpr double kMixedShare = 1.15;   // of a mixed launch's estimate, against the other small tiles', which come out that much high
enum OtherKernel { OTHER_NONE, OTHER_ALIGNED, OTHER_FLEXIBLE, OTHER_SLICED, OTHER_STREAMING };
struct Other {        // what a launch would run else, and for how long by its estimate
    OtherKernel kernel;
    double us;
    bool pipelined;   // a call of the pipelined operator
    bool comm;        // its GEMM launch is followed by a comm launch
};
struct SmallTile {
    int rows, cols;   // 0: the launch is not one for them; 256x256: the large ones of a mixed launch
};
struct SmallTileCost {
    int rows, cols;
    double launch, workgroup, kib, mb, partLine, moved, off16, kn, later;
};
constexpr SmallTileCost kSmallTiles[] = {
    {32, 32, 1.84, 2.42, 0.0118, 0.051, 0.044, 0.234, 0.0049, 0.0053, 0.0},  {32, 64, 2.00, 2.86, 0.0101, 0.079, 0.220, 0.248, 0.0039, 0.0014, 0.0},
    {64, 64, 1.59, 3.86, 0.0120, 0.038, 0.174, 0.238, 0.0033, 0.0010, 0.0},  {64, 128, 3.47, 3.94, 0.0086, 0.187, 0.0, 0.174, 0.0040, 0.0008, 0.0039},
    {96, 128, 3.52, 5.10, 0.0086, 0.213, 0.0, 0.167, 0.0046, 0.0011, 0.0049},  {128, 128, 4.98, 4.59, 0.0085, 0.235, 0.0, 0.185, 0.0045, 0.0010, 0.0051},
    {160, 128, 5.10, 6.26, 0.0093, 0.245, 0.0, 0.190, 0.0042, 0.0011, 0.0053}, {192, 128, 6.15, 6.57, 0.0092, 0.264, 0.0, 0.192, 0.0038, 0.0010, 0.0051}};

struct CallSize {
    double rows, kib, mb, moved;   // rows of the problem, KiB of a row of k, MB of operands, MB of peers and outputs
};

CallSize call_size(const GemmArgs &a, uint32_t es)
{
    const double rows = a.sched.op == OP_ALLGATHER ? (double)a.M * a.sched.P : (double)a.M, kB = (double)a.K * es;
    return {rows, kB / 1024.0, 1e-6 * kB * (a.N + rows), 1e-6 * a.N * (4.0 * a.nPeers * a.keptRows + (a.sched.op == OP_REDUCE_SCATTER ? 4.0 : 2.0) * rows)};
}

// Kept tiles that are spread over all XCDs alike are the first that each of them starts.  Where they run as halves and all workgroups find a slot at once the
// launch takes 0.8 of what others of its size take: of four and eight ranks 150 calls 0.75 to 0.85, W8A8 4096x1280x3072 pipelined 35.5 us (3072x1600x4096, as
// many tiles but not spread alike: 51.5).  With more workgroups eight ranks' take 0.8 to 0.95 (pipelined 2048x1088x8192 as [n,k] 41.0; not 16 bits as [n,k] in
// one round, 4096x1792x4096 87, 83.5 mixed), four ranks' 0.95 to 1.1.
double kept_alike(const GemmArgs &a, bool pipelined)
{
    const uint32_t kept = a.sched.P > 2 ? 8u * splittable_kept_tiles(a) : 0u;
    if (kept == 0) return 1.0;
    if (a.sched.coreLoops + kept <= 512u) return 0.8;
    return a.sched.P >= 8 && (pipelined || !a.transB || a.sched.coreLoops > 512u) ? 0.87 : 1.0;
}

// 128-row tiles of the aligned kernels (launches of 256-row ones run nothing else).
double aligned_us(const GemmArgs &a, uint32_t es, bool pipelined)
{
    const CallSize c = call_size(a, es);
    const double f = a.splitK > 1 ? a.splitK : 1.0, wgs = a.sched.coreLoops * f, rounds = ceil(wgs / 256.0), steps = c.kib * 16.0 / f;
    const double us = 6.6 + rounds * (steps * (0.325 + (a.transB ? 0.060 : 0.0) - (es == 1 ? 0.019 : 0.0)) - 2.0) + (wgs > 512.0 ? 0.104 * (wgs / 256.0 - 2.0) * steps : 0.0) +
                      (f > 1.0 ? 10.0 : 0.0) + (a.sched.op == OP_REDUCE_SCATTER ? 1.88 * a.nPeers : 0.0) + 0.134 * c.moved + 0.505 * c.mb;
    return us * kept_alike(a, pipelined);
}

// Flexible tiles as plan_flex left them in args.fx (blocks = rows / 64): whole, with a second launch for the peers, in k slices.
double flex_us(const GemmArgs &a, uint32_t es, int blocks)
{
    const CallSize c = call_size(a, es);
    const double f = a.fx.slices > 1 ? a.fx.slices : 1.0, wgs = (double)a.fx.rowTiles * a.fx.colTiles * f, rounds = ceil(wgs / 256.0), steps = c.kib * 16.0 / f;
    if (f > 1.0)
        return 9.1 + rounds * steps * (a.transB ? 0.434 : 0.345) + 4e-6 * 0.095 * f * (a.fx.keptOnly ? (double)a.keptRows : c.rows) * a.N + 0.263 * c.moved + 0.112 * c.mb;
    if (a.fx.late) return 8.1 + rounds * steps * (a.transB ? 0.59 : 0.44) + 0.45 * c.moved;
    const double us = 2.5 + rounds * (steps * (0.239 + (a.transB ? 0.126 : 0.0) + (blocks == 2 ? 0.230 : 0.0)) + 3.2) - (wgs > 256.0 ? 0.0855 * wgs / 256.0 * steps : 0.0) +
                      (a.sched.op == OP_REDUCE_SCATTER ? 1.11 * a.nPeers : 0.0) + 0.156 * c.moved + 0.150 * c.mb;
    // (rows of k off the 16-byte grid, many tiles: their copies are bound by the caches)
    const double off16 = blocks == 2 && (uint64_t)a.K * es % 16 != 0 ? wgs / 512.0 * c.kib * 8.0 * (a.transB ? 3.0 : 2.05) + 0.12 * c.moved : 0.0;
    return us > off16 ? us : off16;
}

Other other_flexible(const GemmArgs &a, uint32_t es, int blocks) { return {a.fx.slices > 1 ? OTHER_SLICED : OTHER_FLEXIBLE, flex_us(a, es, blocks), false, false}; }

// Rows of a mixed launch that run on 256x256 tiles, of all but a reduce-scatter's kept ones; `us`: the launch's estimate.
struct MixedRows {
    uint32_t large;
    double us;
};

// A reduce-scatter's kept rows, with their peers, all run on the small tiles; with one rank every row is kept and there are no peers.
bool kept_apart(const GemmArgs &a) { return a.sched.op == OP_REDUCE_SCATTER && a.sched.P > 1; }

// When the last of the workgroups that `cus` CUs get of a launch is done: large ones first, then small ones, each on the first CU that is free.
double part_us(uint64_t large, uint64_t small, double largeUs, double smallUs, uint32_t cus)
{
    const uint32_t parts = 256u / cus;
    const uint64_t l = (large + parts - 1u) / parts, s = (large + small + parts - 1u) / parts - l, part = l % cus, idle = cus - part;
    const double start = (double)(l / cus) * largeUs, end = start + largeUs;   // of the last round of large ones
    if (part == 0) return start + (double)((s + cus - 1u) / cus) * smallUs;
    const uint64_t first = (uint64_t)(largeUs / smallUs) + 1u;   // small ones that a CU without one of those starts by the time they end
    if (s <= idle * first) return fmax(end, start + (double)((s + idle - 1u) / idle) * smallUs);
    const uint64_t left = s - idle * first, more = left / cus, rest = left % cus;
    return fmax(end + (double)(more + (rest ? 1u : 0u)) * smallUs, start + (double)(first + more + (rest > part ? 1u : 0u)) * smallUs);
}

// Two bounds: the CUs' schedule (workgroups go to the XCDs and, mostly, to their four shader engines in turn: the mean of what 32 and
// 8 CUs take) and the power limit, at which large tiles on half of the CUs take less time each than on all.  A small tile's peers come through one CU: the
// fewer small tiles the kept rows are dealt to, the longer each takes.  Fitted to 5953 launches of 899 calls with one to seven counts of rows on large
// tiles each: half of them within 0.04, nine in ten within 0.10; the count with the least estimate takes 1.009 of the best one's time.  Without the peers and with large
// and small tiles rounded up each for itself, so that 253 of them did not fit 256 CUs, it was 1.019 of it, 1.34 at worst: fp16 1800x1344x5888 of eight ranks with stored
// tiles 48.1 -> 38.7 us (161 large and 92 small), W8A8 2440x1728x4224 43.4 -> 36.6, pipelined 4096x1280x3072 as [n,k] 45.3 -> 40.1.
MixedRows mixed_rows(const GemmArgs &a, uint32_t es, uint32_t rows)
{
    const CallSize c = call_size(a, es);
    const double chunks = c.kib * 8.0;
    const bool off16 = (uint64_t)a.K * es % 16 != 0;
    const uint32_t kept = kept_apart(a) ? a.keptRows : 0u;
    const double large = 5.6 + chunks * (off16 ? 1.33 : 1.085) + (kept ? 0.0 : 3.0 * a.nPeers), small = 5.35 + chunks * (off16 ? 0.518 : 0.363) + 0.17 * a.nPeers;
    const uint32_t largeCols = ceil_div(a.N, 256u), smallCols = ceil_div(a.N, 128u), most = ceil_div(rows - kept, 256u);
    // (as few rows on large tiles as leave two rounds of them to the small ones; of a wide range every second, third .. count)
    const uint32_t range = umin(most - 1u, ceil_div(512u, largeCols)), step = range / 32u + 1u;
    MixedRows best = {0, 0.0};
    for (uint32_t t = most - range / step * step; t <= most; t += step) {
        const uint32_t r = umin(256u * t, rows - kept);
        const uint64_t l = (uint64_t)t * largeCols, s = (uint64_t)ceil_div(rows - r, 128u) * smallCols;
        const double dealt = small + (kept ? 0.9 * a.nPeers * kept / (double)(rows - r) : 0.0);
        const double cus = 0.5 * (part_us(l, s, large, dealt, 32u) + part_us(l, s, large, dealt, 8u));
        const double power = 1.36 * chunks * ((double)l + 0.327 * s) / 256.0, c2 = cus * cus, p2 = power * power;
        const double us = sqrt(sqrt(c2 * c2 + p2 * p2));
        if (best.large == 0 || us <= best.us) best = {r, us};
    }
    best.us += 4.4 + 0.108 * c.moved + 0.047 * c.mb;
    return best;
}

void plan_mixed(GemmArgs &a, uint32_t es, uint32_t rows, uint32_t large)
{
    FlexParams &f = a.fx;
    f.rows = large;
    f.rowStep = 256;
    f.perRank = 0;
    f.rowTiles = ceil_div(large, 256u);
    f.colTiles = ceil_div(a.N, 256u);
    f.keptTile0 = f.keptTiles = 0;
    f.tail = (uint32_t)((uint64_t)a.K * es % 128u);
    f.slices = 1;
    f.keptOnly = f.late = 0;
    f.holeRows = rows - large;
    f.keptInHole = kept_apart(a) ? 1u : 0u;
    f.hole0 = f.keptInHole ? umin(a.keptBegin, large) : large;
    f.largeTiles = f.rowTiles * f.colTiles;
}

// Deals a reduce-scatter's kept rows out to the row tiles over `rows` rows (all of them, or those a mixed launch leaves).
void deal_rows(GemmArgs &a, uint32_t es, uint32_t rows, uint32_t tileRows)
{
    const uint32_t tiles = ceil_div(rows, tileRows);
    if (a.sched.op != OP_REDUCE_SCATTER || a.sched.P == 1 || (a.flags & GF_ROW_MASK) || tiles < 2 || (uint64_t)a.M * a.lda * es > 0x7fffffffull) return;
    a.fx.dealRows = rows / tiles;
    a.fx.dealRest = rows % tiles;
    a.fx.dealKept = a.keptRows / tiles;
    a.fx.dealKeptRest = a.keptRows % tiles;
}

// The streaming kernels for explicit kept rows, roughly.
double streaming_us(const GemmArgs &a)
{
    const CallSize c = call_size(a, 1);
    return 9.8 + 1.58e-9 * c.rows * a.K * a.N + 0.147 * c.mb + 0.136 * c.moved + 0.117 * c.kib;
}

// Sliced small tiles: of a row tile that somebody keeps or stores, every slice leaves its partial tile in the workspace.
uint64_t few_partials(const SmallTileCost &t, uint32_t keptTiles, uint32_t n, uint32_t slices) { return (uint64_t)keptTiles * ceil_div(n, (uint32_t)t.cols) * slices * t.rows * t.cols * 4u; }

// A call like those the estimates were compared on (explicit kept rows: any number of ranks).
bool fitted_call(const GemmArgs &a) { return a.N % 32 == 0 && a.K >= 512 && ((a.flags & GF_ROW_MASK) != 0 || (a.sched.P >= 2 && a.sched.P <= 8)); }

// The share of the other kernels' estimate up to which small tiles (wide: of 128 columns; large: mixed ones) run.
double other_share(const GemmArgs &a, uint32_t es, const Other &o, bool sums, bool wide, bool large)
{
    const bool rowMask = (a.flags & GF_ROW_MASK) != 0, rs = a.sched.op == OP_REDUCE_SCATTER;
    if (fitted_call(a)) {
        // (mixed launches, 1400 calls by what would run else: two ranks keep half of all rows, and the other tiles stream the peers under each other's loops; more
        // than 512 aligned tiles, those with a comm launch, flexible ones of k on the 16-byte grid and ragged all-gathers come out shorter than their
        // estimate: pipelined 4096x2880x5120 as [n,k] 79.8 us aligned, 96.8 mixed; two ranks' 4128x1056x3072 37.0 flexible, 43.4)
        if (large) {
            if (!rs) return o.kernel == OTHER_FLEXIBLE && a.sched.op == OP_ALLGATHER ? 0.92 : 1.05;
            if (o.kernel == OTHER_FLEXIBLE) return o.pipelined || (uint64_t)a.K * es % 16 != 0 ? 1.0 : 0.9;
            return a.sched.P == 2 ? 0.92 : a.sched.coreLoops > 512u ? 0.95 : o.comm ? 0.88 : 0.98;
        }
        // (aligned tiles that are all whole, with checksums: they store nothing; 2048x4096x6144 67.5, 76.6 on 128x128; of 450 calls 10 lose more than 0.04, with 1.1 17)
        if (o.kernel == OTHER_ALIGNED && rs && sums && a.sched.P > 2 && a.sched.mRank % a.sched.m0 == 0 && a.N % a.sched.n0 == 0 && kept_alike(a, false) == 1.0) return 1.0;
        // (pipelined calls, a GEMM and a comm launch or one with peers under its loops, come out longer than their estimate, 37 small ones 1.025 -> 1.008 of their
        // best choice's time with 1.1 for 0.95, W8A8 1024x2272x5888 37.7 -> 31.7 us; but none below 640 of k does; two ranks' kept rows are half of all, and aligned tiles then stream
        // peers under each other's loops; the 62 calls with 16-bit operands on whole flexible tiles as [k,n] miss 0.015; with checksums, k on the 16-byte grid, 4520x784x1440 is
        // 28.0 on flexible and 31.3 on 128x128 tiles, off it 2176x6820x4544 133 on flexible and 101 on 160x128; decode calls that could run in k slices, as [k,n], eight ranks 388x7936x512 16.1 there
        // and 18.0 on 32x32 tiles)
        if (o.pipelined) return a.K < 640 ? 0.8 : 1.1;
        if (o.kernel == OTHER_STREAMING) return 0.87;
        if (o.kernel == OTHER_SLICED) return rowMask ? 0.875 : 0.9;
        return o.kernel == OTHER_FLEXIBLE && ((sums && (uint64_t)a.K * es % 16 == 0) || (es == 2 && !a.transB)) ? 0.95 : rs && a.sched.P == 2 ? 1.0 : 1.1;
    }
    double share = o.kernel == OTHER_ALIGNED ? 0.85 : 0.87;
    if (rs && !sums && wide) share *= 1.15;   // (kept rows are dealt out)
    if (!rs && !rowMask) share *= 1.05;
    return o.pipelined ? 0.9 * share : share;
}

// The small tile a launch (operands, schedule, kept rows, flags and pointers filled in) runs, given what would run else;
// fills args.fx for it.  room: the bytes behind the workspace's counter block (a.skCount, if there is one) that the launch may use.
SmallTile small_tile(GemmArgs &a, uint32_t es, const Other &other, uint64_t room = 0)
{
    const SmallTile no = {0, 0};
    const SchedParams &s = a.sched;
    const uint64_t kBytes = (uint64_t)a.K * es, ldaB = (uint64_t)a.lda * es, ldbB = (uint64_t)a.ldb * es;
    const uint64_t rows = s.op == OP_ALLGATHER ? (uint64_t)a.M * s.P : a.M;
    // (4-byte pieces of k; whole 16-byte pieces of a row of B as [k,n]; 32-bit offsets inside a tile)
    if (a.transA || kBytes % 4 != 0 || kBytes < 16 || (!a.transB && ldbB % 16 != 0) || a.N % 4 != 0 || ldaB * 160u > 0x7fffffffull || ldbB * 160u > 0x7fffffffull ||
        rows >= (1u << 30) || s.n0 != 256 || (s.m0 != 64 && s.m0 != 128))
        return no;
    // Checksums: of tasks, and of the 128x128 blocks of explicit kept rows, for tiles that meet in the workspace's counter block (sum_add,
    // sum_in_order) or have all of a block.
    const bool rowMask = (a.flags & GF_ROW_MASK) != 0, sums = (a.flags & GF_OUTBOUND_STORE) == 0 && a.checksum != nullptr && (rowMask || a.keptRows < rows);
    if (sums && !rowMask && (a.skCount == nullptr || s.coreLoops > kCounterBlockBytes / 16u)) return no;
    const CallSize c = call_size(a, es);
    const SmallTileCost *best = nullptr;
    double least = 0.0;
    uint64_t tiles = 0;
    uint32_t slices = 1;
    // (rows nobody keeps leave their sums only)
    const bool keptOnly = rowMask && a.accDump == nullptr;
    auto kept_tile0 = [&](uint32_t step) { return keptOnly ? a.keptBegin / step : 0u; };
    auto kept_tiles = [&](uint32_t step) { return keptOnly ? (a.keptBegin + a.keptRows - 1u) / step + 1u - kept_tile0(step) : (uint32_t)ceil_div((uint32_t)rows, step); };
    // (floats: what a task's tiles add has places of its own there, as many as row tiles can have some of its rows, by column tiles)
    auto sum_parts = [&](const SmallTileCost &t) -> uint32_t {
        const uint32_t dealt = ceil_div((uint32_t)rows, t.rows), h = umin(s.m0, s.mRank);
        const uint32_t least = t.cols != 128 || dealt < 2 ? t.rows : (uint32_t)rows / dealt - a.keptRows / dealt - 1u;   // rows of others that a tile has
        return (int32_t)least < 1 ? 0u : ((h + least - 2u) / least + 1u) * (256u / t.cols);
    };
    const bool fitted = fitted_call(a);
    for (const SmallTileCost &t : kSmallTiles) {
        if (t.cols == 128 && t.rows != 64 && t.rows != 128) {
            // (rows of A and of the peers in 31-bit offsets from a tile's first; the blocks of 128 rows that explicit kept rows' sums are of end where
            // tiles do.  96 rows of an all-reduce or all-gather as [k,n] are not taken, though 58 drawn calls would take 0.94 of their time: 278x4736x4864 of two ranks and
            // 610x4608x5000 of eight are held to the tiles, and so to the bits, that they had)
            if (!fitted || ldaB * t.rows > 0x7fffffffull || (a.nPeers && (uint64_t)a.peerLd * 4u * t.rows > 0x7fffffffull) || (sums && rowMask)) continue;
            if (t.rows == 96 && s.op != OP_REDUCE_SCATTER && !rowMask && !a.transB) continue;
        }
        if (sums && es != 1 && (sum_parts(t) == 0 || s.coreLoops * sum_parts(t) > kCounterBlockBytes / 16u)) continue;
        if (sums && rowMask && (t.cols != 128 || (t.rows < 128 && rows > (uint64_t)t.rows)) && (a.skCount == nullptr || (rows + 127) / 128 * ceil_div(a.N, 128u) > kCounterBlockBytes / 16u))
            continue;
        const uint64_t n = (rows + t.rows - 1) / t.rows * ceil_div(a.N, t.cols);
        if (t.cols < 128 && n > 512) continue;   // (beyond two rounds their operands leave the caches: all-gather 8 x [682,9000] x [9000,672] 234, larger tiles 181)
        // (a second round of 128-wide tiles is a whole one where k is short: the workgroups are mostly start and end. W8A8
        // reduce-scatters of [3320,640] x [640,640] over 4 ranks 15.8 on them, 12.6 on smaller ones; pipelined [3072,512] x [512,768] 15.7, 12.4)
        const double rounds = (double)((n + 255) / 256), perCu = t.cols < 128 || n <= (kBytes <= 1024 ? 512u : 256u) ? rounds : n / 256.0;
        const double perKib = (t.rows + t.cols) * rounds * (t.kib + (kBytes % 16 ? t.off16 : 0.0) + (a.transB ? 0.0 : t.kn) + (n > 256 ? t.later : 0.0));
        const double rest = t.launch + t.workgroup * perCu + c.mb * t.mb + (!a.transB && t.cols * es < 128u ? c.mb * t.partLine : 0.0) + c.moved * t.moved +
                            (sums && !rowMask ? (t.cols == 128 ? 2.0 : 0.7) * rounds + (es != 1 ? 0.5 + 0.05 * sum_parts(t) : 0.0) : 0.0);   // (the tasks' sums)
        for (const uint32_t f : {1u, 2u, 3u, 4u, 6u, 8u}) {
            // (at most a workgroup per CU, two chunks of k per wave; k of whole numbers short enough that their whole sum is within 32 bits, as
            // the slices' sums are that checksums are added up from: 131072 products of -128 and -128 are one past the end)
            if (f > 1 && (t.cols >= 128 || n * f > 256 || kBytes < f * 1024u || (es == 1 && a.K >= 131072u) || a.skCount == nullptr ||
                          few_partials(t, kept_tiles(t.rows), a.N, f) > room))
                break;
            const double us = rest + perKib * c.kib / f + (f > 1 ? 2.2 + 1.5e-4 * f * umin(t.rows, keptOnly ? a.keptRows : (uint32_t)rows) * t.cols : 0.0);
            if (best == nullptr || us < least) {
                best = &t;
                least = us;
                tiles = n;
                slices = f;
            }
        }
    }
    if (best == nullptr) return no;
    // (from three eighths of a round of large tiles on; k in at least a few pairs of steps)
    MixedRows mixed = {0, 0.0};
    if (!sums && rows >= 512 && kBytes >= 1024 && rows * a.N >= 96ull * 256ull * 256ull) {
        mixed = mixed_rows(a, es, (uint32_t)rows);
        if (kMixedShare * mixed.us > least) mixed.large = 0;
    }
    if (other.kernel != OTHER_NONE && (mixed.large ? mixed.us : least) > other_share(a, es, other, sums, mixed.large || best->cols == 128, mixed.large != 0) * other.us) return no;
    if (tiles > (1u << 24) || !flex_ptrs_ok(a)) return no;
    a.fx.dRank = make_fast_div(s.mRank);
    a.splitK = 0;
    if (mixed.large) {
        plan_mixed(a, es, (uint32_t)rows, mixed.large);
        if (a.fx.holeRows) deal_rows(a, es, a.fx.holeRows, 128);
        return {256, 256};
    }
    a.fx.rows = (uint32_t)rows;
    a.fx.rowTiles = (uint32_t)((rows + best->rows - 1) / best->rows);
    a.fx.colTiles = ceil_div(a.N, best->cols);
    a.fx.slices = slices;
    a.fx.keptOnly = keptOnly ? 1u : 0u;
    a.fx.sumParts = sums && es != 1 ? sum_parts(*best) : 0u;
    a.fx.keptTile0 = kept_tile0(best->rows);
    a.fx.keptTiles = kept_tiles(best->rows);
    if (slices > 1) a.skPart = (int32_t *)((unsigned char *)a.skCount + kCounterBlockBytes);
    if (best->cols == 128) deal_rows(a, es, (uint32_t)rows, best->rows);
    return {best->rows, best->cols};
}

int launch_small(uint32_t dtype, const GemmArgs &a, const SmallTile &t, void *stream)
{
    g_launch = {CATCOC_KERNEL_SMALL, (uint32_t)t.rows, (uint32_t)t.cols, t.cols < 128 ? a.fx.slices : 1u, a.fx.dealRows != 0, t.cols == 256 ? a.fx.largeTiles : 0u};
    return t.cols == 256 ? launch_gemm_mixed(dtype, a, stream) : t.cols == 128 ? launch_gemm_mid(dtype, a, t.rows, stream) : launch_gemm_few(dtype, a, t.rows, t.cols, stream);
}

// The workspace's counter block, if the caller gave one.
uint32_t *counter_block(const CatcocSymmetricDesc &d)
{
    return d.workspace != nullptr && (uintptr_t)d.workspace % 256 == 0 && d.workspaceBytes >= kCounterBlockBytes ? (uint32_t *)d.workspace : nullptr;
}

// The bytes behind it that a launch may use whose query says `query`.
uint64_t counter_room(const CatcocSymmetricDesc &d, uint64_t query)
{
    const uint64_t bytes = d.workspaceBytes < query ? d.workspaceBytes : query;
    return counter_block(d) != nullptr && bytes > kCounterBlockBytes ? bytes - kCounterBlockBytes : 0u;
}

// Everything a launcher checks before it launches; fills `plan` except the buffer pointers.
int make_plan(int commType, int dataType, const CocTilingParams *t, const CatcocSymmetricDesc *d, uint32_t transA,
              uint32_t transB, Plan &plan)
{
    if (t == nullptr) return fail(E_NULL, "tiling is NULL");
    if (d == nullptr) return fail(E_NULL, "symmetricPtr is NULL (it must point at a CatcocSymmetricDesc)");
    if (d->magic != CATCOC_DESC_MAGIC) return fail(E_DESC, "symmetricPtr does not point at a CatcocSymmetricDesc (bad magic)");
    if (commType < 0 || commType >= TYPE_NUM) return fail(E_DTYPE, "unknown commType %d", commType);
    const bool quant = commType == QUANT_MATMUL_REDUCE_SCATTER;
    if (quant ? dataType != INT8 : (dataType != FP16 && dataType != BF16))
        return fail(E_DTYPE, "dataType %d is not registered for commType %d", dataType, commType);
    if (t->m == 0 || t->n == 0 || t->k == 0) return fail(E_SHAPE, "empty problem m=%u n=%u k=%u", t->m, t->n, t->k);
    const uint32_t P = d->rankSize;
    if (P == 0 || P > CATCOC_MAX_RANKS) return fail(E_RANK, "rankSize %u out of range 1..%d", P, CATCOC_MAX_RANKS);
    if (t->rankSize != 0 && t->rankSize != P) return fail(E_RANK, "tiling.rankSize %u != descriptor rankSize %u", t->rankSize, P);
    if (d->rankIdx >= P) return fail(E_RANK, "rankIdx %u >= rankSize %u", d->rankIdx, P);

    const uint32_t op = (commType == MATMUL_ALLREDUCE) ? OP_ALLREDUCE : (commType == ALLGATHER_MATMUL) ? OP_ALLGATHER : OP_REDUCE_SCATTER;
    if (op == OP_REDUCE_SCATTER && t->m % P != 0)
        return fail(E_SHAPE, "reduce-scatter needs m %% rankSize == 0 (m=%u, rankSize=%u)", t->m, P);

    const uint32_t blockNum = d->blockNum ? d->blockNum : kDefaultBlockNum;
    const uint32_t stages = d->workspaceStages ? d->workspaceStages : kDefaultStages;
    const uint32_t commInterval = t->commInterval ? t->commInterval : 1u;
    // examples/dynamic_tiling/include/tiling.h:32-41: a round's tiles are dealt evenly to the ranks
    if (op == OP_REDUCE_SCATTER && ((uint64_t)blockNum * commInterval) % P != 0)
        return fail(E_TILING, "blockNum*commInterval = %u*%u is not a multiple of rankSize %u", blockNum, commInterval, P);
    const uint32_t off = d->swizzleOffset ? d->swizzleOffset : 7u;
    const uint32_t dir = d->swizzleOffset ? d->swizzleDirection : 1u;
    if (dir > 1) return fail(E_TILING, "swizzleDirection %u must be 0 or 1", dir);

    const uint32_t dt = (uint32_t)dataType;
    const uint32_t es = elem_size(dt);
    const uint32_t che = 16 / es;
    const uint32_t mRank = op == OP_REDUCE_SCATTER ? t->m / P : t->m;

    // tile selection: the fast kernels have n0 = 256 and m0 in {64,128}, or 256 for W8A8 on full tiles
    uint32_t m0 = t->m0, n0 = t->n0;
    if (n0 == 0) n0 = 256;
    // 256-row tiles: k in whole pairs of 64-byte steps; full tiles, or ragged rows / columns with a whole tile to move an edge
    // tile into and the moved tile's first column on the 16-byte grid of B, D and the peers (as for 128-row tiles below)
    const bool full256 = mRank % 256 == 0 && t->n % 256 == 0;
    const bool can256 = n0 == 256 && !transA && ((uint64_t)t->k * es) % 128 == 0 &&
                        (full256 || (mRank >= 256 && t->n >= 256 && t->n % 8 == 0 && (transB || ((uint64_t)t->n * es) % 16 == 0)));
    if (m0 == 0) {
        // The library's choice: 128-row tiles (two workgroups per CU) unless the launch has at least two 256x256 tiles per CU
        // and a row of k holds 4 KiB or more (or four per CU and 2 KiB): there 256 rows measured 3-10 % faster with B as
        // [k,n] and 15-25 % with B as [n,k] (8192-row launches, both element types, launches alternating); with two tiles
        // per CU and 1792 bytes of k (the benchmark shards) 128 rows stay ahead, 68.8 against 75.7 us.  The
        // rule does not look at the layout of B (with [n,k] the larger tile already pays from 2 KiB of k on): the queries for
        // task counts and workspace sizes do not know the layout and must see the same tiles.  All-gather keeps 128 rows
        // unless the caller asks.
        const uint64_t kBytes = (uint64_t)t->k * es;
        const uint64_t tiles256 = (uint64_t)(t->m / 256u) * (t->n / 256u);
        const bool pays = (tiles256 >= 512 && kBytes >= 4096) || (tiles256 >= 1024 && kBytes >= 2048);
        // (full tiles only: ragged problems take 256 rows on request, since the pipelined operators run those on other kernels)
        m0 = (mRank <= 64) ? 64 : (can256 && full256 && pays && op != OP_ALLGATHER) ? 256 : 128;
    }
    const bool dmaShape = can256 && m0 == 256;
    // (A as [k,m] exists in the 128-row direct-to-LDS kernel only: rows of m in whole 16-byte pieces, a rank's block on that grid)
    const bool taOk = !transA || (m0 == 128 && ((uint64_t)t->m * es) % 16 == 0 && ((uint64_t)mRank * es) % 16 == 0);
    const bool fastShape = dmaShape || n0 == 256 && (m0 == 64 || m0 == 128) && taOk && t->k % che == 0 && t->n % 4 == 0;
    plan.variant = fastShape ? (int)(m0 / 64) : 0;   // 4 (m0 = 256) exists only as the direct-to-LDS kernel
    plan.edge = !(mRank % m0 == 0 && t->n % n0 == 0 && t->k % (64 / es) == 0);
    plan.dtype = dt;
    plan.blockNum = blockNum;
    // (B as [n,k] runs the 128-row direct-to-LDS kernel when its rows of k are 16-byte multiples)
    // Ragged rows / columns on 128-row tiles: the direct-to-LDS kernel moves the edge tiles inwards (GF_RAGGED).  It needs a whole
    // tile to move into, k in whole 64-byte steps, and the moved tile's first column on the 16-byte grid of B, D and the peers.
    const bool ragged = plan.edge && ((m0 == 128 && mRank >= m0 && t->n >= n0 && ((uint64_t)t->k * es) % 64 == 0 && t->n % 8 == 0 &&
                                       (transB || ((uint64_t)t->n * es) % 16 == 0)) ||
                                      (m0 == 256 && can256));
    plan.dma = fastShape && (!plan.edge || ragged) && (m0 == 256 || (m0 == 128 && (!transB || ((uint64_t)t->k * es) % 16 == 0))) &&
               (m0 == 128 || !transA);
    if (transA && !plan.dma) plan.variant = 0;   // the other fast kernels take A as [m,k] only

    GemmArgs &a = plan.args;
    memset(&a, 0, sizeof(a));
    a.M = t->m;
    a.N = t->n;
    a.K = t->k;
    a.lda = transA ? t->m : t->k;
    a.ldb = transB ? t->k : t->n;
    a.ldd = t->n;
    a.transA = transA ? 1 : 0;
    a.transB = transB ? 1 : 0;
    a.outDtype = dt == DT_I8 ? DT_BF16 : dt;
    a.sched = make_sched(op, t->m, t->n, P, m0, n0, blockNum, commInterval, stages, off, dir);
    if (a.sched.coreLoops == 0) return fail(E_SHAPE, "no tiles to compute");

    if ((d->flags & CATCOC_OUTBOUND_MASK) == CATCOC_OUTBOUND_STORE) a.flags |= GF_OUTBOUND_STORE;
    if (d->flags & CATCOC_FLAG_REDUCE_INT32) {
        if (!quant) return fail(E_DESC, "CATCOC_FLAG_REDUCE_INT32 only applies to the W8A8 operator");
        a.flags |= GF_REDUCE_INT32;
    }
    if (d->flags & CATCOC_FLAG_LINEAR_ORDER) a.flags |= GF_LINEAR_ORDER;
    if (d->flags & CATCOC_FLAG_KEPT_WHOLE) a.flags |= GF_KEPT_WHOLE;
    if (d->flags & CATCOC_FLAG_KEPT_SPLIT) a.flags |= GF_KEPT_SPLIT;
    if (plan.dma && plan.edge) a.flags |= GF_RAGGED;

    // kept rows
    if (op == OP_REDUCE_SCATTER) {
        a.keptBegin = d->rankIdx * mRank;
        a.keptRows = mRank;
        a.keptRank = d->rankIdx;
    } else if (op == OP_ALLREDUCE) {
        a.keptBegin = 0;
        a.keptRows = t->m;
    } else {
        a.keptBegin = 0;
        a.keptRows = t->m * P;
    }

    // peers
    const uint32_t nPeers = P - 1;
    if (op == OP_ALLGATHER) {
        a.nPeers = 0;
        uint32_t s = 0;
        for (uint32_t r = 0; r < P; ++r) {
            if (r == d->rankIdx) continue;
            if (d->peers[s] == nullptr) return fail(E_NULL, "all-gather needs %u peer shards; peers[%u] is NULL", nPeers, s);
            a.a[r] = d->peers[s++];
        }
    } else {
        a.nPeers = nPeers;
        for (uint32_t s = 0; s < nPeers; ++s) {
            if (d->peers[s] == nullptr) return fail(E_NULL, "reduce needs %u staged peer partials; peers[%u] is NULL", nPeers, s);
            a.peers[s] = d->peers[s];
        }
        a.peerLd = d->peerLd ? d->peerLd : t->n;
        a.peerRowOffset = d->peerRowOffset;
        if (nPeers && a.peerLd < (int64_t)t->n) return fail(E_DESC, "peerLd %lld < n %u", (long long)a.peerLd, t->n);
        if (a.peerRowOffset < 0) return fail(E_DESC, "peerRowOffset must be >= 0");
        if (fastShape && nPeers && (a.peerLd % 4 != 0)) plan.variant = 0;  // 16-byte peer loads need aligned rows
    }

    if (a.flags & GF_OUTBOUND_STORE) {
        if (op == OP_REDUCE_SCATTER && P > 1) {
            if (d->outbound == nullptr) return fail(E_NULL, "CATCOC_OUTBOUND_STORE needs an outbound buffer");
            const uint64_t need = (uint64_t)stages * a.sched.blockPerComm * m0 * n0 * 4u;
            if (d->outboundBytes < need)
                return fail(E_WORKSPACE, "outbound buffer too small: %llu < %llu bytes", (unsigned long long)d->outboundBytes,
                            (unsigned long long)need);
        }
        a.outbound = d->outbound;
    } else {
        a.checksum = d->checksum;
    }
    a.accDump = d->accDump;

    // Few tiles: the 128-row direct-to-LDS kernel can cut every tile's k range into slices, one workgroup each, that
    // meet through a workspace (partial tiles [tiles][slices][128*256] as 32-bit words, then one counter per tile).
    // Chosen so that the slices fill the 256 CUs once, each with at least eight k steps; float launches take
    // two slices by themselves (see fauto below).  desc.splitK overrides the choice.
    plan.kSlices = 1;
    plan.kSliceBytes = 0;
    if (plan.dma && !plan.edge && m0 == 128 && d->keptRows == 0) {
        const uint32_t T = a.sched.coreLoops, nkAll = (uint32_t)((uint64_t)t->k * es / 64u);
        const uint32_t fmax = 8u;
        // the library's own choice stays at two slices for float operands (more are reproducible too -- three or more float
        // partials are added in slice order -- but did not measure faster: the last slice then fetches every partial)
        const uint32_t fauto = dt == DT_I8 ? 8u : 2u;
        uint32_t f = 1;
        if (d->splitK != 0) {
            if (d->splitK > fmax || d->splitK > nkAll)
                return fail(E_TILING, "splitK %u: at most %u k slices for this k", d->splitK, umin(fmax, nkAll));
            f = d->splitK;
        } else {
            while (f * 2u <= fauto && T * f * 2u <= 256u && nkAll / (f * 2u) >= 8u) f *= 2u;
        }
        if (f > 1) {
            plan.kSlices = f;
            if (T > kMaxCountedTiles) return fail(E_TILING, "k slices: %u tiles exceed the %u the workspace counts", T, kMaxCountedTiles);
            plan.kSliceBytes = kCounterBlockBytes + (uint64_t)T * f * (128u * 256u * 4u);
            if (d->workspace != nullptr) {
                if ((uintptr_t)d->workspace % 256 != 0) return fail(E_WORKSPACE, "workspace must be 256-byte aligned");
                if (d->workspaceBytes < plan.kSliceBytes)
                    return fail(E_WORKSPACE, "workspace too small for %u k slices: %llu < %llu bytes", f,
                                (unsigned long long)d->workspaceBytes, (unsigned long long)plan.kSliceBytes);
                a.splitK = f;
                a.skCount = (uint32_t *)d->workspace;
                a.skPart = (int32_t *)((unsigned char *)d->workspace + kCounterBlockBytes);
            } else if (d->splitK != 0) {
                return fail(E_WORKSPACE, "splitK %u needs a workspace of %llu bytes", f, (unsigned long long)plan.kSliceBytes);
            }
        }
    }
    // Flexible mode takes what the aligned 128- and 256-row kernels do not, and of their launches those whose 64-row tiles leave
    // CUs idle, or fill them once with a short k: twice the workgroups, half the peers per workgroup, k slices that spread the epilogue as well.
    // 128-row tiles (k slices by the library where it takes them) against this, bf16, B as [k,n] / [n,k], launches
    // alternating: 1024x1024x1024 21.1 / 21.8 -> 17.7 / 18.3 us, 1024x4096x1024 37.5 / 40.8 -> 24.6 / 27.3, 1024x1024x4096
    // 27.4 / 28.6 -> 19.8 / 22.4; with seven peers 512x1024x1024 36.7 / 37.4 -> 15.9 / 16.6.  With more tiles, or one per CU and
    // a long k, the larger tile's fewer bytes per product win (2048x4096x4096: 78.5 / 78.8 against 83.6 / 108;
    // 512x8192x8192 in two k slices 93.0 / 102.5 against 111 / 130).  (Checksums stay: a 128-row task would need two workgroups.)
    plan.flexBlocks = 0;
    plan.preferFlex = false;
    plan.maySmall = t->m0 == 0 && d->splitK == 0 && (d->flags & CATCOC_FLAG_LINEAR_ORDER) == 0;
    const uint64_t rowsAll = op == OP_ALLGATHER ? (uint64_t)t->m * P : t->m;
    const uint64_t tiles64 = (rowsAll + 63) / 64 * ceil_div(t->n, 256u);
    const bool fewTiles = tiles64 <= 128u || (tiles64 <= 256u && (uint64_t)t->k * es <= 4096u);
    if (!plan.dma) {
        const FlexSlices c = flex_choose(a, es, t->m0, d->splitK);
        plan.kSlices = c.slices;
        plan.kSliceBytes = c.bytes;
        plan.flexBlocks = flex_use(a, es, t->m0, c, d->workspace, d->workspaceBytes);
    } else if (m0 == 128 && t->m0 == 0 && (d->splitK == 0 || (plan.edge && d->splitK > 1)) && (d->flags & CATCOC_FLAG_LINEAR_ORDER) == 0 && fewTiles && !transA &&
               !(op == OP_REDUCE_SCATTER && P > 1 && a.checksum != nullptr)) {
        // What a workspace takes is said for the aligned kernel, and this one uses the slices that fit into that, unless it would
        // take four or more: all-reduce of 257x14336x512, bf16, seven peers, in 64 KiB of workspace (no slices) / in what its slices
        // take: 156 / 21 us; 306x13824x2048 147 / 41; reduce-scatter 832x15232x800 of four ranks with stored tiles 157 / 52.
        // (Rows of B that end inside a 16-byte piece have an aligned kernel as [n,k] only: the query speaks of flexible tiles.)
        // Ragged rows or columns have k slices here only, so a caller's own count of them is for this kernel.
        const FlexSlices c = flex_choose(a, es, 0, d->splitK);
        plan.preferFlex = c.whole != 0;
        if (plan.preferFlex && ((c.slices >= 4 && c.bytes > plan.kSliceBytes) || ((uint64_t)t->n * es) % 16 != 0 || d->splitK > 1)) {
            if (plan.kSlices == 1) plan.kSlices = c.slices;   // (the aligned kernel's count is what launches with A as [k,m] run)
            plan.kSliceBytes = c.bytes;
        }
        plan.flexBlocks = flex_use(a, es, 0, c, d->workspace, d->workspaceBytes < plan.kSliceBytes ? d->workspaceBytes : plan.kSliceBytes);
        // A reduce-scatter that gets neither slices nor a second launch for its peers, and whose kept tiles the aligned kernel runs as
        // two workgroups each: there the halves shorten the same chain without the flexible tiles' set-up.  Aligned / flexible tiles,
        // stored tiles, no workspace, us: k of 1 KiB or less, W8A8 512x512x4096 of four ranks 9.6 / 11.3, fp16 1024x512x4096 of two
        // 11.7 / 13.5 (2 KiB: 512x2048x4096 17.3 / 17.3, 16 bits 512x1024x4096 16.0 / 15.2); more than 128 tiles, W8A8 2048x2048x2048 of
        // eight ranks 25.9 / 27.8, as [n,k] 26.1 / 29.5, of four 19.5 / 22.8, 20.1 / 24.3, k = 4096 29.9 / 32.0, 35.2 / 36.2, of eight
        // 35.9 / 37.2, 41.6 / 41.5; with one peer and B as [k,n] the larger k is the flexible tiles' (768x4096x4096 28.9 / 26.7).
        // (The caller's choice between halves and whole tiles does not enter: keep_aligned.)
        const uint64_t kBytes = (uint64_t)t->k * es;
        const uint32_t flags = a.flags;
        a.flags &= ~(uint32_t)(GF_KEPT_WHOLE | GF_KEPT_SPLIT);
        if (plan.preferFlex && op == OP_REDUCE_SCATTER && a.fx.slices <= 1 && a.fx.late == 0 &&
            (kBytes <= 1024 || (tiles64 > 128u && (kBytes <= 2048 || nPeers > 1 || transB))) && split_kept_tiles(a, (uint32_t)(kBytes / 64)) != 0)
            plan.preferFlex = false;
        a.flags = flags;
        // (Floats on ragged rows or columns, B as [k,n], four slices or more: these run the count that the query reports, so that a caller who names it
        // has the bits of one who leaves it open.  All others may run small tiles, which add in another order.  What that holds back, flexible /
        // small tiles, us, operands in the caches, bf16 all-reduce of eight ranks: 257x4096x512 14.3 / 9.9, 300x2048x1032 15.8 / 10.0, 131x8192x1288 17.8 / 19.6.  Whole numbers
        // are the same in any order: W8A8 290x2496x736 12.7 -> 7.7, two ranks 500x3776x640 15.1 -> 9.2, 30 calls take 0.58 to 0.97 of their time)
        if (plan.preferFlex && plan.edge && !transB && es != 1 && a.fx.slices >= 4) plan.maySmall = false;
    }
    plan.counters = counter_block(*d);
    plan.room = counter_room(*d, plan.kSliceBytes);
    // a workspace also lets the checksum halves of tiles that run as two workgroups meet (its counter block)
    if (a.skCount == nullptr && d->workspace != nullptr && (uintptr_t)d->workspace % 256 == 0 && d->workspaceBytes >= kCounterBlockBytes)
        a.skCount = (uint32_t *)d->workspace;
    if (d->flags & CATCOC_FLAG_TAIL_WHOLE) a.flags |= GF_TAIL_WHOLE;
    return 0;
}

int check_ptr_align(const Plan &p, const void *a, const void *b)
{
    if (p.variant == 0) return 1;
    const uint32_t es = elem_size(p.dtype);
    bool okA = ((uintptr_t)a % 16 == 0) && ((p.args.lda * es) % 16 == 0);
    bool okB = p.args.transB ? (((uintptr_t)b % 16 == 0) && ((p.args.ldb * es) % 16 == 0))
                             : (((uintptr_t)b % (4 * es) == 0) && (p.args.ldb % 4 == 0));
    for (uint32_t r = 0; r < p.args.sched.P && okA; ++r)
        if (p.args.a[r] && (uintptr_t)p.args.a[r] % 16 != 0) okA = false;
    return okA && okB;
}

// The small tile that a planned launch runs, if any (g: its arguments); dma, flex: what it would run else.
SmallTile planned_small(const Plan &p, bool dma, bool flex, GemmArgs &g)
{
    if (!p.maySmall) return {0, 0};
    g = p.args;
    // Whole tiles of other ranks that are neither stored nor summed: no operator's use, but what tools ask about and time (catcoc_kept_split_tiles,
    // catcoc_launch_tile); these launches run the tiles and the order that the queries know.
    if ((dma || p.preferFlex) && (g.flags & GF_OUTBOUND_STORE) == 0 && g.checksum == nullptr && g.sched.op == OP_REDUCE_SCATTER && splittable_kept_tiles(g) != 0) return {0, 0};
    g.skCount = p.counters;
    const uint32_t es = elem_size(p.dtype);
    return small_tile(g, es, dma ? Other{OTHER_ALIGNED, aligned_us(p.args, es, false), false, false} : flex ? other_flexible(p.args, es, p.flexBlocks) : Other{OTHER_NONE, 0.0, false, false}, p.room);
}

// CATCOC_FLAG_KEPT_WHOLE and CATCOC_FLAG_KEPT_SPLIT change no bit of a result: sums of floats in another order would.  So they do not enter the
// choice of small tiles or of k slices, and only move a launch of whole flexible tiles, which add in the aligned kernel's order, there.
bool keep_aligned(const GemmArgs &a) { return (a.flags & (GF_KEPT_WHOLE | GF_KEPT_SPLIT)) != 0 && a.fx.slices <= 1 && splittable_kept_tiles(a) != 0; }

bool launched_small(const Plan &p, bool dma, bool flex, void *stream)
{
    GemmArgs g;
    const SmallTile t = planned_small(p, dma, flex, g);
    if (t.rows) launched(launch_small(p.dtype, g, t, stream));
    return t.rows != 0;
}

void launch_float(int commType, int dataType, void *stream, uint8_t *a, uint8_t *b, uint8_t *c, uint8_t *symmetricPtr,
                  CocTilingParams *tiling, uint32_t transA, uint32_t transB)
{
    Plan p;
    const CatcocSymmetricDesc *d = (const CatcocSymmetricDesc *)symmetricPtr;
    if (make_plan(commType, dataType, tiling, d, transA, transB, p)) return;
    if (!a || !b || !c) { fail(E_NULL, "a, b and c must be non-NULL"); return; }
    if (commType == ALLGATHER_MATMUL) p.args.a[d->rankIdx] = a;
    else p.args.a[0] = a;
    p.args.b = b;
    p.args.d = c;
    if (!check_ptr_align(p, a, b)) p.variant = 0;
    const bool preferFlex = p.preferFlex && flex_ptrs_ok(p.args);
    const bool aligned = p.dma && p.variant != 0 && (uintptr_t)b % 16 == 0 && (p.args.ldb * 2) % 16 == 0 && (uintptr_t)c % 16 == 0;
    bool dma = !preferFlex && aligned;
    if (!dma) p.args.splitK = 0;   // the other kernels run every tile whole
    if (!dma && p.variant == 4) { fail(E_TILING, "m0 = 256 needs full tiles and 16-byte aligned row-major operands"); return; }
    if (!dma && p.args.transA) p.variant = 0;
    const bool flex = !dma && p.flexBlocks != 0 && flex_ptrs_ok(p.args);
    if (launched_small(p, dma, flex, stream)) return;
    if (aligned && keep_aligned(p.args)) dma = true;
    const int e = dma ? launch_gemm_dma(p.dtype, p.args, stream)
                  : flex ? launch_flex(p.dtype, p.args, p.flexBlocks, stream)
                      : launch_gemm(p.dtype, p.args, p.variant, p.edge, stream);
    if (e) { fail(E_LAUNCH, "kernel launch failed: %s", hipGetErrorString((hipError_t)e)); return; }
    ok();
}

// ---- skinny-M split-K path (explicit kept rows) ----------------------------------------------
struct SplitkPlan {
    GemmArgs args;
    uint32_t f, tiles, rowBlocks;
    uint64_t workspaceBytes;   // partial tiles + counters (0 when f == 1)
    bool general = false;      // shape outside the fast routes: flexible mode, or gemm_general_kernel on the 128x128 grid
    int flexBlocks;            // (general) as Plan::flexBlocks
    bool preferFlex;           // sliced row tiles (flexible mode) run although the streaming kernels would take the launch
    bool maySmall;             // as Plan::maySmall
    bool wholeK;               // at most 32 rows against B as [n,k]: gemm_decode_nk_kernel, no k slices, no workspace
    bool large;                // many rows: the 128x256 direct-to-LDS kernel in row-mask mode runs instead of the split-K kernel
};

// Explicit kept rows with at least this many rows of A run the 128x256 direct-to-LDS kernel (k-sliced through the same
// workspace) when the shape has full tiles and the kept rows are whole 32-row blocks.  Such launches have at most one
// workgroup per CU and run the kernel's six-stage ring with the pipelined peer loads.  Measured at K = N = 8192 with kept
// rows = M / 8, the two routes alternating launch by launch and B coming from HBM (six copies, another one every launch):
// M = 1024 106 against 166 us, M = 512 69 (two k slices) against 77 us, M = 256 50 (four k slices) against 48 us (since then
// both routes fetch A as whole cache lines per pair of k steps and hand only kept blocks between k slices: M = 512 59 against 74 us,
// M = 384 56 against 103 (three rows of 128x128 tiles in four slices are three waves of workgroups), M = 256 42 against 50, and with
// 32 kept rows M = 128 45 (eight k slices) against 36, so the large tile starts at 256 rows).  n0 = 256
// (with m0 0 or 128) in the tiling asks for the large tile explicitly, n0 = 128 for the split-K kernel.
constexpr uint32_t kLargeTileRows = 256;

int make_splitk_plan(const CocTilingParams *t, const CatcocSymmetricDesc *d, uint32_t transA, uint32_t transB, SplitkPlan &sp)
{
    if (t == nullptr) return fail(E_NULL, "tiling is NULL");
    if (d == nullptr || d->magic != CATCOC_DESC_MAGIC) return fail(E_DESC, "symmetricPtr does not point at a CatcocSymmetricDesc");
    if (t->m == 0 || t->n == 0 || t->k == 0) return fail(E_SHAPE, "empty problem m=%u n=%u k=%u", t->m, t->n, t->k);
    const uint32_t P = d->rankSize;
    if (P == 0 || P > CATCOC_MAX_RANKS) return fail(E_RANK, "rankSize %u out of range 1..%d", P, CATCOC_MAX_RANKS);
    if (transA) return fail(E_SHAPE, "the explicit-kept-rows (split-K) path takes A as [m,k] (B as [k,n] or, with transB, as [n,k])");
    // shapes the two fast routes cannot take (k not in whole 64-byte steps, n not in whole 128-column tiles) run small or
    // flexible tiles where k and n are multiples of four, else the one-thread-per-element kernel on the 128x128 grid, a correctness path:
    // whole tiles and nothing behind the counter block either way
    sp.general = t->k % 64 != 0 || t->n % 128 != 0;
    sp.wholeK = false;
    sp.preferFlex = false;
    sp.maySmall = t->m0 == 0 && t->n0 == 0 && d->splitK == 0 && d->blockNum == 0;
    const bool canLarge = !sp.general && t->m % 128 == 0 && t->n % 256 == 0 && d->keptRowBegin % 32 == 0 && d->keptRows % 32 == 0;
    const bool wantLarge = t->n0 == 256 && (t->m0 == 0 || t->m0 == 128);
    if (wantLarge && !canLarge)
        return fail(E_TILING, "128x256 tiles with explicit kept rows need m %% 128 == 0, n %% 256 == 0 and kept rows in whole 32-row blocks "
                              "(m=%u, n=%u, kept [%u,+%u))", t->m, t->n, d->keptRowBegin, d->keptRows);
    sp.large = wantLarge || (t->n0 == 0 && t->m0 == 0 && canLarge && t->m >= kLargeTileRows);
    if (!sp.large && ((t->m0 != 0 && t->m0 != 128) || (t->n0 != 0 && t->n0 != 128)))
        return fail(E_TILING, "explicit kept rows run 128x128 tiles (split-K kernel) or 128x256 tiles; leave m0/n0 zero or pass one of those "
                              "(m0=%u, n0=%u)", t->m0, t->n0);
    if (d->keptRows == 0 || (uint64_t)d->keptRowBegin + d->keptRows > t->m)
        return fail(E_DESC, "kept rows [%u,+%u) outside [0,%u)", d->keptRowBegin, d->keptRows, t->m);
    if ((d->flags & CATCOC_OUTBOUND_MASK) == CATCOC_OUTBOUND_STORE)
        return fail(E_DESC, "the split-K path folds non-kept rows into checksums; CATCOC_OUTBOUND_STORE is not supported there");
    const uint32_t off = d->swizzleOffset ? d->swizzleOffset : 7u;
    const uint32_t dir = d->swizzleOffset ? d->swizzleDirection : 1u;
    if (dir > 1) return fail(E_TILING, "swizzleDirection %u must be 0 or 1", dir);

    GemmArgs &a = sp.args;
    memset(&a, 0, sizeof(a));
    a.M = t->m; a.N = t->n; a.K = t->k;
    a.lda = t->k; a.ldb = transB ? t->k : t->n; a.ldd = t->n;
    a.transB = transB ? 1 : 0;
    if (d->flags & CATCOC_FLAG_REDUCE_INT32) a.flags |= GF_REDUCE_INT32;   // int32 peers join the accumulators before the dequant
    a.outDtype = DT_BF16;
    a.sched.off = off; a.sched.dir = dir;
    a.keptBegin = d->keptRowBegin;
    a.keptRows = d->keptRows;
    a.nPeers = P - 1;
    for (uint32_t s = 0; s < a.nPeers; ++s) {
        if (d->peers[s] == nullptr) return fail(E_NULL, "reduce needs %u staged peer partials; peers[%u] is NULL", a.nPeers, s);
        a.peers[s] = d->peers[s];
    }
    a.peerLd = d->peerLd ? d->peerLd : t->n;
    a.peerRowOffset = d->peerRowOffset;
    if (a.nPeers && a.peerLd < (int64_t)t->n) return fail(E_DESC, "peerLd %lld < n %u", (long long)a.peerLd, t->n);
    if (a.peerRowOffset < 0) return fail(E_DESC, "peerRowOffset must be >= 0");
    if ((uint64_t)(a.peerRowOffset + a.keptRows) * (uint64_t)a.peerLd * 4u > 0x7fffffffull)
        return fail(E_DESC, "the split-K path addresses each peer partial with 31-bit byte offsets: (peerRowOffset + keptRows) * peerLd * 4 must stay below 2 GiB");
    a.checksum = d->checksum;
    a.accDump = d->accDump;

    const uint32_t cores = d->blockNum ? d->blockNum : kDefaultBlockNum;
    const uint32_t kTiles = ceil_div(t->k, 256u);
    sp.tiles = ceil_div(t->m, 128u) * ceil_div(t->n, 128u);
    if (sp.general) {
        if (d->splitK > 1) return fail(E_TILING, "k %% 64 != 0 or n %% 128 != 0: this shape runs whole tiles on the general kernels; splitK %u is not available", d->splitK);
        const uint32_t stages = d->workspaceStages ? d->workspaceStages : kDefaultStages;
        a.sched = make_sched(OP_ALLREDUCE, t->m, t->n, 1, 128, 256, cores, 1, stages, off, dir);
        a.flags |= GF_ROW_MASK;
        sp.rowBlocks = 4;
        // (whole tiles: the query asks for no workspace; of one that is there small tiles use the counter block, for sums that meet)
        sp.flexBlocks = plan_flex(a, 1, a.checksum != nullptr, 0, 1);
        sp.f = 1;
        sp.workspaceBytes = 0;
        if (sp.flexBlocks == 0) a.sched = make_sched(OP_ALLREDUCE, t->m, t->n, 1, 128, 128, cores, 1, stages, off, dir);
        a.splitK = 0;
        return 0;
    }
    // Flexible mode (gemm_flex.h) where its 64-row tiles in k slices beat the streaming kernels: those hand a tile's slices and
    // all its peers to one workgroup, the flexible launch spreads both over every CU, and of rows that are not kept it stores no
    // partial sums.  Streaming kernels -> this, W8A8, seven peers, all rows kept unless said, launches alternating, us:
    // 203x1792x4096 37.9 -> 18.5, 128x8192x1024 46.3 -> 15.0, 512x1024x1024 29.0 -> 14.1, 64x8192x8192 30.1 -> 24.5 (8 rows kept
    // 22.7 -> 19.9), 203x8192x8192 56.6 -> 40.1, 16x8192x2048 with 2 rows kept 16.1 -> 13.1.  The other way round:
    //  - weights of more than 64 MiB stream better through the deep rings of those kernels (64x16384x8192 42.0 / 43.5, as [n,k]
    //    44.8 / 53.8; 388x15744x5376 94 / 111);
    //  - at most 32 rows with a k that leaves nothing to slice, or little to win: a second launch costs 1 us (17x576x896 10.0 / 11.2,
    //    8x1024x8192 10.4 / 10.1, 2x8192x8192 with one row kept, [n,k], 18.2 / 19.3), or with so many columns that partial sums of
    //    more than a few kept rows outweigh the rest (24x4096x8192 13.9 / 15.8, 12x4608x7168 of eight ranks, [n,k], 1.11 times;
    //    with 5120 or 6144 columns 0.9-1.0 as [k,n], 1.02-1.11 as [n,k]);
    //  - many rows in full tiles, few of them kept: the 128x256 tile's fewer bytes per product (512x8192x8192 with 64 rows kept
    //    50 / 65, 512x4096x8192 with 256 rows kept 35 / 40, 256x8192x8192 and one peer 43.4 / 45.5).
    if (t->m0 == 0 && t->n0 == 0 && d->splitK == 0 && d->blockNum == 0) {
        const uint64_t weights = (uint64_t)t->k * t->n, work64 = (uint64_t)ceil_div(t->m, 64u) * ceil_div(t->n, 256u) * t->k;
        sp.preferFlex = t->m <= 32 ? t->k >= 4096 && weights <= (32ull << 20) && t->n <= (transB && d->keptRows > t->m / 4 ? 4096u : 6144u)
                                   : weights <= (64ull << 20) && (!sp.large || work64 <= 128u * 4096u || (d->keptRows == t->m && P > 2));
    }
    if (sp.large) {
        // one grid of 128x256 tiles over all of A's rows (no rank structure), k slices as for any few-tile launch
        const uint32_t stages = d->workspaceStages ? d->workspaceStages : kDefaultStages;
        a.sched = make_sched(OP_ALLREDUCE, t->m, t->n, 1, 128, 256, cores, 1, stages, off, dir);
        a.flags |= GF_ROW_MASK;
        const uint32_t T = a.sched.coreLoops, nkAll = t->k / 64u;
        uint32_t f = 1;
        if (d->splitK != 0) {
            if (d->splitK > 8u || d->splitK > nkAll) return fail(E_TILING, "splitK %u: at most %u k slices here", d->splitK, umin(8u, nkAll));
            f = d->splitK;
        } else {
            while (f * 2u <= 8u && T * f * 2u <= 256u && nkAll / (f * 2u) >= 8u) f *= 2u;
        }
        if (f > 1 && T > kMaxCountedTiles) return fail(E_TILING, "k slices: %u tiles exceed the %u the workspace counts", T, kMaxCountedTiles);
        sp.f = f;
        a.splitK = f > 1 ? f : 0;
        sp.rowBlocks = 4;
        sp.workspaceBytes = f > 1 ? kCounterBlockBytes + (uint64_t)T * f * (128u * 256u * 4u) : 0;
        return 0;
    }
    // B as [n,k] against at most 32 rows: a workgroup can own 32 columns over the whole k range and still read whole cache
    // lines, so nothing is handed between workgroups (unless the caller asks for k slices or for per-tile checksums, which
    // are per 128 columns)
    sp.wholeK = transB && t->m <= 32 && t->k % 128 == 0 && d->splitK <= 1 && d->checksum == nullptr;
    if (sp.wholeK) {
        sp.f = 1;
        a.splitK = 0;
        sp.rowBlocks = 1;
        sp.workspaceBytes = 0;
        return 0;
    }
    uint32_t f = d->splitK ? d->splitK : splitk_factor(t->m, t->n, t->k, cores, 128, 128, 256);
    if (f > kTiles) f = kTiles;
    if (f == 0) f = 1;
    sp.f = f;
    a.splitK = f;
    sp.rowBlocks = t->m <= 32 ? 1 : t->m <= 64 ? 2 : 4;
    if (f > 1 && sp.tiles > kMaxCountedTiles)
        return fail(E_TILING, "split-K: %u tiles exceed the %u the workspace counts", sp.tiles, kMaxCountedTiles);
    sp.workspaceBytes = f > 1 ? kCounterBlockBytes + (uint64_t)f * sp.tiles * 128u * 128u * 4u : 0;
    return 0;
}

// Launches with explicit kept rows that preferFlex leaves to the streaming kernels all the same, by what only a planned launch
// says.  Streaming / flexible, W8A8, us, B as [k,n] unless said:
//  - whole tiles with checksums are 128 rows high, and one workgroup has all of a kept tile's peers: 128x256x2048 with 16 rows
//    kept of eight ranks 10.9 / 22.7, of one 9.8 / 12.8, 512x512x8192 with 128 kept 25.7 / 27.4, 203x4096x16384 with 25 kept
//    33.7 / 45.3 (the other way up to 1 KiB of k where the streaming kernels would slice or run more than one round:
//    64x448x4096 of two ranks 12.3 / 11.3, 300x1024x16384 of eight 25.0 / 21.3);
//  - whole tiles without, k too short for slices: few kept rows (64x192x4096 with 8 kept of eight ranks 8.5 / 13.6, 256x192x4096
//    with 32 kept 11.6 / 15.4), all of fewer than 48 rows with several peers (33x256x2048 11.5 / 12.8); with half the rows kept,
//    64 at least, the flexible tiles win (128x192x4096 with 64 kept 14.6 / 12.0);
//  - full 128x256 tiles, one peer at most: more 64-row tiles than CUs (384x1024x16384 with 96 kept of one rank 13.3 / 15.6), and a
//    long k without peers where two slices leave CUs idle or B is [n,k] (384x4096x4096 23.8 / 25.9, 512x4096x4096 [n,k]
//    26.8 / 29.8).
bool decode_flex_pays(const GemmArgs &g, bool large)
{
    const uint32_t tiles64 = ceil_div(g.M, 64u) * g.fx.colTiles;
    if (large && g.nPeers <= 1 && tiles64 > 256u) return false;
    if (large && g.nPeers == 0 && g.keptRows == g.M && g.K >= 4096 && tiles64 > 64u && (tiles64 <= 96u || g.transB)) return false;
    if (g.fx.slices >= 2) return true;
    if (g.checksum != nullptr) return !large && g.K > 256 && g.K <= 1024 && (g.nPeers <= 1 || g.K >= 512);
    if (g.K >= 512) return true;
    if (g.keptRows == g.M) return g.M >= 48 || g.nPeers <= 1;
    if (g.keptRows >= 64 && g.keptRows >= g.M - g.keptRows) return true;
    return !large && (g.K > 256 ? g.nPeers <= 1 || g.M >= 128 : g.nPeers == 0);
}

void launch_quant_splitk(void *stream, uint8_t *x1, uint8_t *x2, uint8_t *scale_x1, uint8_t *scale_x2, uint8_t *bias,
                         uint8_t *c_accum, uint8_t *d_out, const CatcocSymmetricDesc *d, CocTilingParams *tiling,
                         uint32_t transA, uint32_t transB, uint32_t outDataType)
{
    SplitkPlan sp;
    if (make_splitk_plan(tiling, d, transA, transB, sp)) return;
    if (!x1 || !x2 || !scale_x1 || !scale_x2 || !d_out) { fail(E_NULL, "x1, x2, scale_x1, scale_x2 and d_out must be non-NULL"); return; }
    if (outDataType != FP16 && outDataType != BF16) { fail(E_DTYPE, "outDataType %u must be FP16 (1) or BF16 (27)", outDataType); return; }
    GemmArgs &a = sp.args;
    if (sp.general) {
        a.a[0] = x1; a.b = x2; a.d = d_out;
        a.scaleM = (const float *)scale_x1; a.scaleN = (const float *)scale_x2;
        a.bias = (const int32_t *)bias; a.cAccum = (int32_t *)c_accum;
        a.outDtype = outDataType;
        if (sp.maySmall) {   // (the rest of these shapes runs whole 64x256 tiles or one thread per element, many times slower)
            GemmArgs g = a;
            g.skCount = counter_block(*d);
            const SmallTile t = small_tile(g, 1, {OTHER_NONE, 0.0, false, false});
            if (t.rows) { launched(launch_small(DT_I8, g, t, stream)); return; }
        }
        const bool flex = sp.flexBlocks != 0 && flex_ptrs_ok(a);
        if (!flex && a.sched.n0 != 128) {
            const SchedParams &g = a.sched;
            a.sched = make_sched(OP_ALLREDUCE, a.M, a.N, 1, 128, 128, g.blockPerComm, 1, g.stages, g.off, g.dir);
        }
        const int eg = flex ? launch_flex(DT_I8, a, sp.flexBlocks, stream) : launch_gemm(DT_I8, a, 0, true, stream);
        if (eg) { fail(E_LAUNCH, "kernel launch failed: %s", hipGetErrorString((hipError_t)eg)); return; }
        ok();
        return;
    }
    if ((uintptr_t)x1 % 16 != 0 || (uintptr_t)x2 % 16 != 0 || sp.args.lda % 16 != 0 || sp.args.ldb % 16 != 0) {
        fail(E_SHAPE, "the split-K path needs 16-byte aligned x1, x2 and row pitches");
        return;
    }
    // The large-tile route picked its k slices by itself (no desc.splitK): they need a workspace to meet through, and without
    // one that fits the tiles run whole, as any other few-tile launch of that kernel does.  Only an explicit splitK insists.
    if (sp.large && sp.f > 1 && d->splitK == 0 &&
        (d->workspace == nullptr || (uintptr_t)d->workspace % 256 != 0 || d->workspaceBytes < sp.workspaceBytes)) {
        sp.f = 1;
        a.splitK = 0;
    }
    if (sp.f > 1) {
        if (d->workspace == nullptr || d->workspaceBytes < sp.workspaceBytes) {
            fail(E_WORKSPACE, "split factor %u needs a zero-initialised workspace of %llu bytes (catcoc_get_splitk_workspace_size)",
                 sp.f, (unsigned long long)sp.workspaceBytes);
            return;
        }
        if ((uintptr_t)d->workspace % 256 != 0) { fail(E_WORKSPACE, "workspace must be 256-byte aligned"); return; }
        a.skCount = (uint32_t *)d->workspace;
        a.skPart = (int32_t *)((unsigned char *)d->workspace + kCounterBlockBytes);
    }
    a.a[0] = x1;
    a.b = x2;
    a.d = d_out;
    a.scaleM = (const float *)scale_x1;
    a.scaleN = (const float *)scale_x2;
    a.bias = (const int32_t *)bias;
    a.cAccum = (int32_t *)c_accum;
    a.outDtype = outDataType;
    // The plan above says what the launch is refused for and what it asks of the workspace, whichever kernel runs.
    const auto flex = [&]() {
        // (few rows of a long k and few columns as [n,k]: the whole-k kernel's rings for up to eight rows hold more of B than a 32x32
        // tile's.  Whole k / small tiles, us: 8x16384x2048 13.3 / 13.9, 1x12288x1024 10.8 / 11.5, 1x8192x512 8.6 / 9.0; not 8x8192x2048 10.2 / 9.6,
        // 8x12288x3072 13.6 / 11.9, 1x8192x8192 16.0 / 15.1, 16x4096x8192 10.6 / 9.4.  And weights that stay in the cache, where a long k is a chain
        // of waits: eight ranks, 12x16384x512 with 2 rows kept 12.1 / 13.0, 16x24576x256 with 2 16.5 / 17.4, 9x32768x128 with all 18.7 / 21.3, 8x12288x512
        // with one 10.3 / 10.8.  All else of 9 to 32 rows is small tiles': calls with k of 4096 to 32768 and n of 128 to 8192 take 0.74 to 1.05 of
        // the whole-k kernel's time, 20x32768x256 with 3 rows kept 1.07.)
        const bool few = 4u * a.keptRows <= a.M, cached = (uint64_t)a.K * a.N <= (10u << 20);
        const bool deepK = sp.wholeK && (a.M <= 4 ? a.K >= 8192 && a.N <= (a.K > 8192 ? 4096u : 2048u) : a.M <= 8 ? a.K > (few && cached ? 11264u : 12288u) && a.N <= 2048 :
                                         a.M <= 16 && cached && a.K >= (few ? 14336u : 24576u));
        if (deepK || (!sp.maySmall && !sp.preferFlex)) return false;
        GemmArgs g = a;
        const uint32_t stages = d->workspaceStages ? d->workspaceStages : kDefaultStages;
        g.sched = make_sched(OP_ALLREDUCE, a.M, a.N, 1, 128, 256, kDefaultBlockNum, 1, stages, a.sched.off, a.sched.dir);
        g.flags |= GF_ROW_MASK;
        g.splitK = 0;
        g.skCount = nullptr;
        GemmArgs small = g;
        small.skCount = counter_block(*d);
        int blocks = 0;
        if (sp.preferFlex && !sp.wholeK) {
            const FlexSlices c = flex_choose(g, 1, 0, 0);
            blocks = flex_use(g, 1, 0, c, d->workspace, d->workspaceBytes < sp.workspaceBytes ? d->workspaceBytes : sp.workspaceBytes);
            // (without the slices it would take, only where the streaming kernels run whole tiles as well)
            if ((c.slices > 1 && g.fx.slices < 2 && (sp.large || sp.f > 1)) || !decode_flex_pays(g, sp.large) || !flex_ptrs_ok(g)) blocks = 0;
        }
        if (sp.maySmall) {
            const SmallTile t = small_tile(small, 1, sp.wholeK ? Other{OTHER_NONE, 0.0, false, false} : blocks ? other_flexible(g, 1, blocks) : Other{OTHER_STREAMING, streaming_us(g), false, false},
                                           counter_room(*d, sp.workspaceBytes));
            // (a call that takes the kept rows' int32 block as well and would run in k slices runs in k slices, of one kind or the other: what its
            // workspace query reports is held to be what runs there.  Whole small tiles would be faster: operands in the caches, 203x1792x4096 with
            // all rows kept 18.5 / 10.8 us, 512x1024x1024 of two ranks 12.8 / 6.3)
            const bool sliced = blocks ? g.fx.slices > 1 : sp.f > 1;
            if (t.rows && !(a.cAccum != nullptr && sliced && small.fx.slices <= 1)) {
                launched(launch_small(DT_I8, small, t, stream));
                return true;
            }
        }
        if (blocks == 0) return false;
        const int e = launch_flex(DT_I8, g, blocks, stream);
        if (e) fail(E_LAUNCH, "kernel launch failed: %s", hipGetErrorString((hipError_t)e));
        else ok();
        return true;
    };
    if (sp.large) {
        bool aligned = (uintptr_t)scale_x2 % 16 == 0 && (uintptr_t)d_out % 16 == 0 && (!bias || (uintptr_t)bias % 16 == 0) && a.peerLd % 4 == 0;
        for (uint32_t s = 0; s < a.nPeers && aligned; ++s) aligned = (uintptr_t)a.peers[s] % 16 == 0;
        if (!aligned) { fail(E_SHAPE, "128x256 tiles with explicit kept rows need 16-byte aligned scales, bias, peers and output"); return; }
        if (flex()) return;
        const int el = launch_gemm_dma(DT_I8, a, stream);
        if (el) { fail(E_LAUNCH, "kernel launch failed: %s", hipGetErrorString((hipError_t)el)); return; }
        ok();
        return;
    }
    if (flex()) return;
    g_launch = {CATCOC_KERNEL_STREAMING, sp.wholeK ? 32u : 128u, sp.wholeK ? 32u : 128u, sp.f, 0, 0};
    const int e = sp.wholeK ? launch_gemm_decode_nk_i8(a, stream) : launch_gemm_splitk_i8(a, (int)sp.rowBlocks, sp.tiles * sp.f, stream);
    if (e) { fail(E_LAUNCH, "kernel launch failed: %s", hipGetErrorString((hipError_t)e)); return; }
    ok();
}

void launch_quant(void *stream, uint8_t *x1, uint8_t *x2, uint8_t *scale_x1, uint8_t *scale_x2, uint8_t *bias,
                  uint8_t *c_accum, uint8_t *d_out, uint8_t *symmetricPtr, CocTilingParams *tiling, uint32_t transA,
                  uint32_t transB, uint32_t outDataType)
{
    Plan p;
    const CatcocSymmetricDesc *d = (const CatcocSymmetricDesc *)symmetricPtr;
    if (d != nullptr && d->magic == CATCOC_DESC_MAGIC && d->keptRows != 0) {
        launch_quant_splitk(stream, x1, x2, scale_x1, scale_x2, bias, c_accum, d_out, d, tiling, transA, transB, outDataType);
        return;
    }
    if (make_plan(QUANT_MATMUL_REDUCE_SCATTER, INT8, tiling, d, transA, transB, p)) return;
    if (!x1 || !x2 || !scale_x1 || !scale_x2 || !d_out) { fail(E_NULL, "x1, x2, scale_x1, scale_x2 and d_out must be non-NULL"); return; }
    if (outDataType != FP16 && outDataType != BF16) { fail(E_DTYPE, "outDataType %u must be FP16 (1) or BF16 (27)", outDataType); return; }
    p.args.a[0] = x1;
    p.args.b = x2;
    p.args.d = d_out;
    p.args.scaleM = (const float *)scale_x1;
    p.args.scaleN = (const float *)scale_x2;
    p.args.bias = (const int32_t *)bias;
    p.args.cAccum = (int32_t *)c_accum;
    p.args.outDtype = outDataType;
    if (!check_ptr_align(p, x1, x2) || (uintptr_t)scale_x2 % 16 != 0 || (bias && (uintptr_t)bias % 16 != 0) ||
        (c_accum && (uintptr_t)c_accum % 16 != 0) || (uintptr_t)d_out % 8 != 0)
        p.variant = 0;
    const bool preferFlex = p.preferFlex && flex_ptrs_ok(p.args);
    bool aligned = p.dma && p.variant != 0 && (uintptr_t)x2 % 16 == 0 && p.args.ldb % 16 == 0 && (uintptr_t)d_out % 16 == 0;
    for (uint32_t s = 0; s < p.args.nPeers && aligned; ++s) aligned = (uintptr_t)p.args.peers[s] % 16 == 0;
    bool dma = !preferFlex && aligned;
    if (!dma && p.variant == 4) { fail(E_TILING, "m0 = 256 needs full tiles, 16-byte aligned row-major operands and fp32 peers"); return; }
    if (!dma) p.args.splitK = 0;   // the other kernels run every tile whole
    if (!dma && p.args.transA) p.variant = 0;
    const bool flex = !dma && p.flexBlocks != 0 && flex_ptrs_ok(p.args);
    if (launched_small(p, dma, flex, stream)) return;
    if (aligned && keep_aligned(p.args)) dma = true;
    const int e = dma ? launch_gemm_dma(p.dtype, p.args, stream) : flex ? launch_flex(p.dtype, p.args, p.flexBlocks, stream) : launch_gemm(p.dtype, p.args, p.variant, p.edge, stream);
    if (e) { fail(E_LAUNCH, "kernel launch failed: %s", hipGetErrorString((hipError_t)e)); return; }
    ok();
}

}  // namespace

// The events of a round-pipelined call: "store finished" and "compute finished" per round, and the join at the end.
struct CatcocPipelinedPlan {
    uint32_t magic = 0;
    std::vector<hipEvent_t> ready, done;
    hipEvent_t fin = nullptr;
};

namespace {

constexpr uint32_t kPlanMagic = 0x4350504cu;   // "CPPL"

void plan_destroy_events(CatcocPipelinedPlan &p)
{
    for (hipEvent_t e : p.ready) if (e) (void)hipEventDestroy(e);
    for (hipEvent_t e : p.done) if (e) (void)hipEventDestroy(e);
    if (p.fin) (void)hipEventDestroy(p.fin);
    p.ready.clear();
    p.done.clear();
    p.fin = nullptr;
    p.magic = 0;
}

bool plan_make_events(CatcocPipelinedPlan &p, uint32_t rounds)
{
    p.ready.assign(rounds, nullptr);
    p.done.assign(rounds, nullptr);
    hipError_t he = hipEventCreateWithFlags(&p.fin, hipEventDisableTiming);
    for (uint32_t r = 0; r < rounds && he == hipSuccess; ++r) {
        he = hipEventCreateWithFlags(&p.ready[r], hipEventDisableTiming);
        if (he == hipSuccess) he = hipEventCreateWithFlags(&p.done[r], hipEventDisableTiming);
    }
    if (he != hipSuccess) {
        plan_destroy_events(p);
        fail(E_LAUNCH, "hipEventCreate failed: %s", hipGetErrorString(he));
        return false;
    }
    p.magic = kPlanMagic;
    return true;
}

// ---- round-pipelined, reference-faithful form of the reduce-scatter operators ------------------
// The reference's structure kept as it is (quant_matmul_reduce_scatter.hpp:159-164,219,282,319; matmul_reduce_scatter.hpp
// the same): per comm round the GEMM stores the round's tiles (kept rank's into the local block, the others into stage
// `round % stages` of the workspace) and raises "store finished"; the comm side waits for it, adds the peers' blocks into
// the local block along BlockCommSwizzle's task list and raises "compute finished", which the GEMM of round + stages
// waits for before it reuses the stage.  The two sides are two HIP streams here and the flags are events.
void launch_pipelined(bool quant, int dataType, void *computeStream, void *commStream, uint8_t *a, uint8_t *b, uint8_t *scale_x1,
                      uint8_t *scale_x2, uint8_t *bias, uint8_t *c_accum, uint8_t *d_out, uint8_t *symmetricPtr,
                      CocTilingParams *tiling, uint32_t transA, uint32_t transB, uint32_t outDataType, uint32_t deterministic)
{
    const CatcocSymmetricDesc *given = (const CatcocSymmetricDesc *)symmetricPtr;
    if (given == nullptr || given->magic != CATCOC_DESC_MAGIC) { fail(E_DESC, "symmetricPtr does not point at a CatcocSymmetricDesc"); return; }
    if (given->keptRows != 0) { fail(E_DESC, "the round-pipelined form keeps the reference's row blocks (keptRows must be 0)"); return; }
    CatcocSymmetricDesc d = *given;
    d.flags = (d.flags & ~CATCOC_OUTBOUND_MASK) | CATCOC_OUTBOUND_STORE | CATCOC_FLAG_LINEAR_ORDER;
    if (quant) d.flags |= CATCOC_FLAG_REDUCE_INT32;
    d.workspace = nullptr;
    d.splitK = 0;
    Plan p;
    const int commType = quant ? QUANT_MATMUL_REDUCE_SCATTER : MATMUL_REDUCE_SCATTER;
    if (make_plan(commType, dataType, tiling, &d, transA, transB, p)) return;
    if (!a || !b || !d_out) { fail(E_NULL, "operands and output must be non-NULL"); return; }
    if (quant && (!scale_x1 || !scale_x2 || !c_accum)) { fail(E_NULL, "the pipelined W8A8 operator needs scale_x1, scale_x2 and c_accum"); return; }
    const uint32_t outDt = quant ? outDataType : (uint32_t)dataType;
    if (outDt != FP16 && outDt != BF16) { fail(E_DTYPE, "outDataType %u must be FP16 (1) or BF16 (27)", outDt); return; }
    if (d.outbound == nullptr && d.rankSize > 1) { fail(E_NULL, "the pipelined form stores the other ranks' tiles: outbound (the symmetric workspace) is needed"); return; }

    GemmArgs &g = p.args;
    const SchedParams &sp = g.sched;
    const uint32_t P = sp.P, m0 = sp.m0, n0 = sp.n0;
    const uint32_t cb = tiling->commBlockM ? tiling->commBlockM : umin(64u, m0);
    if (m0 % cb != 0) { fail(E_TILING, "commBlockM %u must divide m0 %u", cb, m0); return; }
    uint32_t splitRow = tiling->commDataSplit, splitCol = tiling->commNpuSplit ? tiling->commNpuSplit : 1u;
    if (splitRow == 0 || splitRow * splitCol < 16u) { splitRow = 256u; splitCol = 1u; }   // the reference's 2..20 cores would idle this GPU
    if (!deterministic && P % splitCol != 0) { fail(E_TILING, "commNpuSplit %u must divide rankSize %u", splitCol, P); return; }
    const uint32_t es = quant ? 4u : 2u;
    const uint32_t vec = 16u / es;
    if (tiling->n % vec != 0 || n0 % vec != 0) { fail(E_SHAPE, "the pipelined form moves 16-byte pieces: n and n0 must be multiples of %u", vec); return; }
    const int64_t peerLd = d.peerLd ? d.peerLd : tiling->n;
    void *local = quant ? (void *)c_accum : (void *)d_out;
    if ((uintptr_t)local % 16 != 0 || (peerLd * es) % 16 != 0) { fail(E_SHAPE, "the pipelined form needs 16-byte aligned blocks and peer rows"); return; }
    for (uint32_t s = 0; s + 1 < P; ++s)
        if ((uintptr_t)d.peers[s] % 16 != 0) { fail(E_SHAPE, "peers[%u] must be 16-byte aligned", s); return; }

    // GEMM side: every round is one launch of the ordinary kernels over the round's tasks, with no peers to add
    if (quant) {
        g.a[0] = a; g.b = b; g.d = d_out;
        g.scaleM = (const float *)scale_x1; g.scaleN = (const float *)scale_x2;
        g.bias = (const int32_t *)bias; g.cAccum = (int32_t *)c_accum;
        g.outDtype = outDt;
        if (!check_ptr_align(p, a, b) || (uintptr_t)scale_x2 % 16 != 0 || (bias && (uintptr_t)bias % 16 != 0) || (uintptr_t)d_out % 8 != 0) p.variant = 0;
    } else {
        g.a[0] = a; g.b = b; g.d = d_out;
        if (!check_ptr_align(p, a, b)) p.variant = 0;
    }
    g.nPeers = 0;
    const bool dma = p.dma && !p.edge && p.variant != 0 && (uintptr_t)b % 16 == 0 && (g.ldb * (quant ? 1 : 2)) % 16 == 0 && (uintptr_t)d_out % 16 == 0;
    g.flags &= ~(uint32_t)GF_RAGGED;   // (ragged problems run the bounds-checked kernel here)
    if (!dma && p.variant == 4) { fail(E_TILING, "m0 = 256 needs full tiles and 16-byte aligned row-major operands"); return; }
    if (!dma && g.transA) p.variant = 0;
    // A call of one round is one launch over all tasks: it runs in flexible mode what the aligned kernels do not take (ragged rows
    // or columns, which otherwise meet a bounds-checked kernel with hundreds of spilled registers) and few tiles of a short k, as
    // the fused operators do.  W8A8, GEMM launch and comm launch, us: 2048x1792x1440 53.6 -> 27.6, 1536x3904x640 88.0 -> 29.3;
    // aligned 1024x1792x2048 27.4 -> 25.6, 512x8192x4096 58.3 -> 45.2 (512x576x4096 18.0 / 18.4: not below 1 KiB of k).
    int flexBlocks = 0;
    if (sp.coreLoops <= sp.blockPerComm) {
        const uint32_t es1 = quant ? 1u : 2u;
        const uint64_t tiles64 = (uint64_t)ceil_div(tiling->m, 64u) * ceil_div(tiling->n, 256u);
        if (!dma || (m0 == 128 && !transA && (uint64_t)tiling->k * es1 >= 1024u && (tiles64 <= 128u || (tiles64 <= 256u && (uint64_t)tiling->k * es1 <= 4096u))))
            flexBlocks = plan_flex(g, es1, false, 0, 1);
        if (flexBlocks != 0 && !flex_ptrs_ok(g)) flexBlocks = 0;
    }
    // A W8A8 call of one round on aligned tiles has no round to overlap its comm launch with, and int32 sums come out the same in
    // any order: the fused operator's epilogue adds the peers, under the other tiles' main loops, and one launch writes tiles, sums
    // and output.  That hides the peers (nPeers x 128 KiB through the CU of a kept tile) where workgroups are still waiting for a slot,
    // where half the CUs are free and kept tiles run as halves, and where the peers are few; in between the second launch's
    // stream over every CU is shorter than the chain it replaces.  Two launches -> one, us, launches alternating: 512 tiles of eight ranks
    // 4096x1792x4096 55.2 -> 48.3, as [n,k] 58.8 -> 50.2, 384 tiles 3072x1024x8192 61.3 -> 55.5, 128 tiles 1024x8192x4096 73.4 -> 61.7, two
    // ranks 4096x4096x2048 58.3 -> 50.9, four 2048x512x4096 24.6 -> 21.0; not 288 tiles of eight 2048x2048x4608 47.6 -> 56.3, 256 of
    // four 2048x4096x4096 52.8 -> 59.8.
    const bool oneRound = sp.coreLoops <= sp.blockPerComm;
    bool fused = quant && dma && flexBlocks == 0 && P > 1 && oneRound &&
                 (sp.coreLoops >= 384u || sp.coreLoops <= 128u || P == 2 || (P <= 4 && tiling->k <= 2048u));
    if (fused) g.nPeers = P - 1;
    // (a single round may run in the order of the fused operators: 4096x8192x8192 of two ranks, as [n,k], two launches 405 -> 337)
    if (oneRound && (given->flags & CATCOC_FLAG_LINEAR_ORDER) == 0) g.flags &= ~(uint32_t)GF_LINEAR_ORDER;
    // Small or mixed tiles do the same in one launch, for problems of any alignment.  The fused operator's choice, with the comm launch on the
    // other side where it is not fused.  GEMM and comm launch -> one, us, one row-block round of eight ranks: 1024x3904x768 40.4 ->
    // 16.3, 2048x10672x1024 68.8 -> 38.7, 3072x2304x6176 91.5 -> 70.9, 4096x8960x7072 325 -> 280, of four 512x3604x640 45.0 -> 11.8, of two
    // 1792x6784x1024 49.7 -> 24.7; the other way round 4096x1792x4096 48.9 / 59.7, 3072x576x1792 24.1 / 26.6.
    SmallTile small = {0, 0};
    GemmArgs gs = g;
    if (quant && P > 1 && oneRound && (given->flags & (CATCOC_FLAG_LINEAR_ORDER | CATCOC_FLAG_KEPT_WHOLE | CATCOC_FLAG_KEPT_SPLIT)) == 0) {
        const double comm = fused ? 0.0 : 4.5 + 0.8 * (P - 1) + 0.1e-6 * 4.0 * (P - 1) * g.keptRows * g.N;
        gs.nPeers = P - 1;
        small = small_tile(gs, 1, flexBlocks ? Other{OTHER_FLEXIBLE, flex_us(g, 1, flexBlocks) + comm, true, true} : dma ? Other{OTHER_ALIGNED, aligned_us(g, 1, true) + comm, true, !fused} : Other{OTHER_NONE, 0.0, false, false});
    }
    if (small.rows) fused = true;
    const bool commWritesOutput = quant && !fused && deterministic != 0 && P > 1 && (uintptr_t)scale_x2 % 16 == 0 && (uintptr_t)d_out % 8 == 0;
    if ((dma || flexBlocks) && commWritesOutput) g.flags |= GF_KEPT_INT32_ONLY;   // (the comm rounds write every kept row's output)

    CommArgs c;
    memset(&c, 0, sizeof(c));
    c.local = local;
    c.localLd = tiling->n;
    for (uint32_t s = 0; s + 1 < P; ++s) c.peers[s] = d.peers[s];
    c.peerLd = peerLd;
    c.peerRowOffset = d.peerRowOffset;
    c.P = P; c.rank = d.rankIdx;
    c.mRank = sp.mRank; c.N = tiling->n;
    c.m0 = m0; c.n0 = n0; c.loopsM = sp.loopsM; c.loopsN = sp.loopsN; c.off = sp.off; c.dir = sp.dir;
    c.commBlockM = cb;
    c.splitRow = splitRow; c.splitCol = splitCol;
    c.swizzleDir = 0;
    c.dtype = quant ? (uint32_t)CT_INT32 : outDt;
    const uint32_t cores = splitRow * splitCol;
    // deterministic W8A8 rounds finish their blocks themselves (int32 sums and the dequantised rows in one pass over them)
    const bool fuseDequant = commWritesOutput;
    if (fuseDequant) {
        c.dOut = d_out;
        c.ldd = tiling->n;
        c.scaleN = (const float *)scale_x2;
        c.scaleM = (const float *)scale_x1 + (size_t)d.rankIdx * sp.mRank;
        c.outDtype = outDt;
    }

    const uint32_t bpc = sp.blockPerComm, perRank = bpc / P, stages = sp.stages;
    const uint32_t rounds = ceil_div(sp.coreLoops, bpc);
    // the events: the caller's plan, or a set made for this call alone
    CatcocPipelinedPlan own;
    CatcocPipelinedPlan *plan = given->pipelinedPlan;
    if (plan != nullptr) {
        if (plan->magic != kPlanMagic) { fail(E_DESC, "desc.pipelinedPlan does not point at a CatcocPipelinedPlan"); return; }
        if (plan->ready.size() < rounds) {
            fail(E_WORKSPACE, "this call has %u comm rounds; the plan holds events for %u", rounds, (uint32_t)plan->ready.size());
            return;
        }
    } else if (rounds > 1 && computeStream != commStream) {   // (a single round, or one stream, needs no event)
        plan = &own;
        if (!plan_make_events(own, rounds)) return;
    } else {
        plan = &own;
        own.ready.assign(rounds, nullptr);
        own.done.assign(rounds, nullptr);
    }
    std::vector<hipEvent_t> &ready = plan->ready, &done = plan->done;
    hipEvent_t fin = plan->fin;
    auto destroy = [&]() { if (plan == &own) plan_destroy_events(own); };
    hipError_t he = hipSuccess;
    // A single round has nothing to overlap: its comm side then runs on computeStream behind the GEMM and no event is needed.
    const bool oneStream = rounds == 1 || computeStream == commStream;
    hipStream_t cs = (hipStream_t)computeStream, ms = oneStream ? cs : (hipStream_t)commStream;
    int e = 0;
    for (uint32_t r = 0; r < rounds && e == 0 && he == hipSuccess; ++r) {
        const uint32_t first = r * bpc, actual = umin(bpc, sp.coreLoops - first);
        if (r >= stages && !oneStream) he = hipStreamWaitEvent(cs, done[r - stages], 0);   // "compute finished" of the stage's last user
        g.taskBase = first;
        g.taskCount = oneRound ? 0 : actual;
        if (he == hipSuccess)
            e = small.rows ? launch_small(p.dtype, gs, small, computeStream)
                : flexBlocks ? launch_flex(p.dtype, g, flexBlocks, computeStream)
                : dma ? launch_gemm_dma(p.dtype, g, computeStream)
                    : launch_gemm(p.dtype, g, p.variant, p.edge, computeStream);
        if (e == 0 && he == hipSuccess && !oneStream) he = hipEventRecord(ready[r], cs);   // "store finished"
        if (e == 0 && he == hipSuccess && !oneStream) he = hipStreamWaitEvent(ms, ready[r], 0);
        c.roundFirstIdx = r * perRank;
        c.dataLoops = (actual / P) * (m0 / cb);
        if (e == 0 && he == hipSuccess && P > 1 && c.dataLoops > 0 && !fused) e = launch_comm_reduce(c, cores, deterministic != 0, ms);
        if (e == 0 && he == hipSuccess && !oneStream) he = hipEventRecord(done[r], ms);
    }
    if (e == 0 && he == hipSuccess && quant && !fuseDequant && !fused)   // the pass after all rounds: dequantise the reduced int32 block
        e = launch_dequant_rows((const int32_t *)c_accum, tiling->n, (const float *)scale_x2, (const float *)scale_x1 + (size_t)d.rankIdx * sp.mRank,
                                d_out, tiling->n, sp.mRank, tiling->n, outDt, ms);
    if (e == 0 && he == hipSuccess && !oneStream) he = hipEventRecord(fin, ms);
    if (e == 0 && he == hipSuccess && !oneStream) he = hipStreamWaitEvent(cs, fin, 0);   // the caller's stream sees the finished output
    destroy();
    if (e) { fail(E_LAUNCH, "kernel launch failed: %s", hipGetErrorString((hipError_t)e)); return; }
    if (he != hipSuccess) { fail(E_LAUNCH, "stream/event call failed: %s", hipGetErrorString(he)); return; }
    ok();
}

// ---- built-in scratch for callers that cannot allocate ---------------------------------------
// One array per GPU, part of the library's code object: it exists from the moment the library is loaded on a device
// until the process ends.  In host code the array's name is only a handle for hipGetSymbolAddress; everything that
// needs the memory (kernel arguments, the fill below) uses the per-device address obtained from it.
static __device__ __align__(256) unsigned char scratch[CATCOC_STATIC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
struct ScratchState { void *ptr; };
ScratchState g_scratch[kMaxDevices];
pthread_mutex_t g_scratchLock = PTHREAD_MUTEX_INITIALIZER;

// Address of the current device's copy of `scratch`; NULL on failure.  Nothing has to be cleared: a __device__ array is
// zero when the code object is loaded, and every launch leaves the counter block at zero again for the next.
void *scratch_for_current_device()
{
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        fail(E_LAUNCH, "no current HIP device (or more than %d devices)", kMaxDevices);
        return nullptr;
    }
    pthread_mutex_lock(&g_scratchLock);
    ScratchState &st = g_scratch[dev];
    if (st.ptr == nullptr) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || p == nullptr) {
            pthread_mutex_unlock(&g_scratchLock);
            fail(E_LAUNCH, "hipGetSymbolAddress(scratch) failed on device %d: %s", dev, hipGetErrorString(e));
            return nullptr;
        }
        st.ptr = p;
    }
    void *p = st.ptr;
    pthread_mutex_unlock(&g_scratchLock);
    return p;
}

}  // namespace

extern "C" {

void catcoc_launch_quant_matmul_reduce_scatter_static_scratch(void *stream, uint64_t fftsAddr, uint8_t *x1, uint8_t *x2,
                                                              uint8_t *scale_x1, uint8_t *scale_x2, uint8_t *bias,
                                                              uint8_t *c_accum, uint8_t *d_out, uint8_t *symmetricPtr,
                                                              CocTilingParams *tiling, uint32_t transA, uint32_t transB,
                                                              uint32_t outDataType)
{
    (void)fftsAddr;
    const CatcocSymmetricDesc *given = (const CatcocSymmetricDesc *)symmetricPtr;
    if (given == nullptr || given->magic != CATCOC_DESC_MAGIC) {
        fail(E_DESC, "symmetricPtr does not point at a CatcocSymmetricDesc");
        return;
    }
    CatcocSymmetricDesc d = *given;
    d.workspace = nullptr;
    d.workspaceBytes = 0;
    // how much scratch would this launch use?  Plan it first, with the sizes only.
    uint64_t need = 0;
    bool optional = false;   // (launches in flexible mode take the k slices that fit)
    {
        CatcocSymmetricDesc q = d;
        for (int i = 0; i < CATCOC_MAX_RANKS; ++i) if (!q.peers[i]) q.peers[i] = (const void *)16;
        if (q.keptRows != 0) {
            SplitkPlan sp;
            if (make_splitk_plan(tiling, &q, transA, transB, sp)) return;
            need = sp.workspaceBytes;
        } else {
            Plan p;
            if ((q.flags & CATCOC_OUTBOUND_MASK) == CATCOC_OUTBOUND_STORE) q.checksum = nullptr;   // (the launch will not look at it)
            q.flags &= ~CATCOC_OUTBOUND_MASK;
            if (make_plan(QUANT_MATMUL_REDUCE_SCATTER, INT8, tiling, &q, transA, transB, p)) return;
            need = p.kSliceBytes;
            optional = p.flexBlocks != 0;
        }
    }
    if (optional) need = need < (uint64_t)CATCOC_STATIC_SCRATCH_BYTES ? need : (uint64_t)CATCOC_STATIC_SCRATCH_BYTES;
    if (need > (uint64_t)CATCOC_STATIC_SCRATCH_BYTES) {
        fail(E_WORKSPACE, "this launch needs %llu bytes of scratch; the built-in scratch holds %llu "
                          "(use catcoc_launch_quant_matmul_reduce_scatter with a workspace of your own)",
             (unsigned long long)need, (unsigned long long)CATCOC_STATIC_SCRATCH_BYTES);
        return;
    }
    if (need != 0) {
        void *p = scratch_for_current_device();
        if (p == nullptr) return;
        d.workspace = p;
        d.workspaceBytes = CATCOC_STATIC_SCRATCH_BYTES;
    }
    launch_quant(stream, x1, x2, scale_x1, scale_x2, bias, c_accum, d_out, (uint8_t *)&d, tiling, transA, transB, outDataType);
}

#define FLOAT_LAUNCHER(name, commType, dataType)                                                                      \
    void name(void *stream, uint64_t fftsAddr, uint8_t *a, uint8_t *b, uint8_t *c, uint8_t *aW, uint8_t *bW,           \
              uint8_t *symmetricPtr, CocTilingParams *tiling, uint32_t transA, uint32_t transB)                        \
    {                                                                                                                  \
        (void)fftsAddr; (void)aW; (void)bW;                                                                            \
        launch_float(commType, dataType, stream, a, b, c, symmetricPtr, tiling, transA, transB);                       \
    }

FLOAT_LAUNCHER(catcoc_launch_matmul_allreduce_fp16, MATMUL_ALLREDUCE, FP16)
FLOAT_LAUNCHER(catcoc_launch_matmul_allreduce_bf16, MATMUL_ALLREDUCE, BF16)
FLOAT_LAUNCHER(catcoc_launch_allgather_matmul_fp16, ALLGATHER_MATMUL, FP16)
FLOAT_LAUNCHER(catcoc_launch_allgather_matmul_bf16, ALLGATHER_MATMUL, BF16)
FLOAT_LAUNCHER(catcoc_launch_matmul_reduce_scatter_fp16, MATMUL_REDUCE_SCATTER, FP16)
FLOAT_LAUNCHER(catcoc_launch_matmul_reduce_scatter_bf16, MATMUL_REDUCE_SCATTER, BF16)

CatcocKernelFuncPtr catcoc_get_kernel(int commType, int dataType)
{
    switch ((commType << 8) | dataType) {  // key of KernelDispatcher::Hash, launch_map.h:30-33
        case (MATMUL_ALLREDUCE << 8) | FP16: return catcoc_launch_matmul_allreduce_fp16;
        case (MATMUL_ALLREDUCE << 8) | BF16: return catcoc_launch_matmul_allreduce_bf16;
        case (ALLGATHER_MATMUL << 8) | FP16: return catcoc_launch_allgather_matmul_fp16;
        case (ALLGATHER_MATMUL << 8) | BF16: return catcoc_launch_allgather_matmul_bf16;
        case (MATMUL_REDUCE_SCATTER << 8) | FP16: return catcoc_launch_matmul_reduce_scatter_fp16;
        case (MATMUL_REDUCE_SCATTER << 8) | BF16: return catcoc_launch_matmul_reduce_scatter_bf16;
        default: return nullptr;
    }
}

void catcoc_launch_quant_matmul_reduce_scatter(void *stream, uint64_t fftsAddr, uint8_t *x1, uint8_t *x2,
                                               uint8_t *scale_x1, uint8_t *scale_x2, uint8_t *bias, uint8_t *c_accum,
                                               uint8_t *d_out, uint8_t *symmetricPtr, CocTilingParams *tiling,
                                               uint32_t transA, uint32_t transB, uint32_t outDataType)
{
    (void)fftsAddr;
    launch_quant(stream, x1, x2, scale_x1, scale_x2, bias, c_accum, d_out, symmetricPtr, tiling, transA, transB, outDataType);
}

void catcoc_quant_matmul_reduce_scatter(void *stream, uint64_t fftsAddr, uint8_t *x1, uint8_t *x2, uint8_t *scale_x1,
                                        uint8_t *scale_x2, uint8_t *bias, uint8_t *c_accum, uint8_t *d_out,
                                        uint8_t *symmetricPtr, uint32_t m, uint32_t n, uint32_t k)
{
    (void)fftsAddr;
    // the example's fixed configuration (quant_matmul_reduce_scatter.cpp:93-147): tile 128x256, commInterval 10
    CocTilingParams t;
    memset(&t, 0, sizeof(t));
    t.m = m; t.n = n; t.k = k;
    t.m0 = 128; t.n0 = 256; t.k0 = 256;
    t.commInterval = 10;
    t.commTileM = 64; t.commBlockM = 64; t.commNpuSplit = 1; t.commDataSplit = 20;
    const CatcocSymmetricDesc *d = (const CatcocSymmetricDesc *)symmetricPtr;
    t.rankSize = (d && d->magic == CATCOC_DESC_MAGIC) ? d->rankSize : 0;
    launch_quant(stream, x1, x2, scale_x1, scale_x2, bias, c_accum, d_out, symmetricPtr, &t, 0, 0, BF16);
}

const char *catcoc_last_error(void) { return g_err; }
int catcoc_last_status(void) { return g_status; }

int catcoc_can_implement(int commType, int dataType, const CocTilingParams *tiling, const CatcocSymmetricDesc *desc,
                         uint32_t transA, uint32_t transB)
{
    Plan p;
    const int e = make_plan(commType, dataType, tiling, desc, transA, transB, p);
    if (!e) ok();
    return e;
}

uint64_t catcoc_get_workspace_size(int commType, int dataType, const CocTilingParams *tiling, const CatcocSymmetricDesc *desc)
{
    Plan p;
    CatcocSymmetricDesc d;
    if (desc == nullptr || tiling == nullptr) { fail(E_NULL, "tiling and desc must be non-NULL"); return 0; }
    d = *desc;
    d.flags &= ~CATCOC_OUTBOUND_MASK;  // size query must not require the buffer it sizes
    for (int i = 0; i < CATCOC_MAX_RANKS; ++i) if (!d.peers[i]) d.peers[i] = (const void *)16;
    if (make_plan(commType, dataType, tiling, &d, 0, 0, p)) return 0;
    ok();
    return (uint64_t)p.args.sched.stages * p.args.sched.blockPerComm * p.args.sched.m0 * p.args.sched.n0 * 4u;
}

uint64_t catcoc_get_kslice_workspace_size(int commType, int dataType, const CocTilingParams *tiling, const CatcocSymmetricDesc *desc,
                                          uint32_t *kSlices)
{
    Plan p;
    CatcocSymmetricDesc d;
    if (desc == nullptr || tiling == nullptr) { fail(E_NULL, "tiling and desc must be non-NULL"); return 0; }
    d = *desc;
    if ((d.flags & CATCOC_OUTBOUND_MASK) == CATCOC_OUTBOUND_STORE) d.checksum = nullptr;   // (the launch will not look at it)
    d.flags &= ~CATCOC_OUTBOUND_MASK;
    d.workspace = nullptr;
    const uint32_t forced = d.splitK;
    d.splitK = 0;
    for (int i = 0; i < CATCOC_MAX_RANKS; ++i) if (!d.peers[i]) d.peers[i] = (const void *)16;
    if (forced != 0) {   // size for the caller's own slice count: plan it with a workspace that is large enough
        d.splitK = forced;
        d.workspace = (void *)256;
        d.workspaceBytes = ~0ull;
    }
    if (make_plan(commType, dataType, tiling, &d, 0, 0, p)) return 0;
    ok();
    if (kSlices) *kSlices = p.kSlices;
    return p.kSliceBytes;
}

uint64_t catcoc_get_splitk_workspace_size(const CocTilingParams *tiling, const CatcocSymmetricDesc *desc, uint32_t *splitK,
                                          uint32_t *tiles)
{
    SplitkPlan sp;
    CatcocSymmetricDesc d;
    if (desc == nullptr || tiling == nullptr) { fail(E_NULL, "tiling and desc must be non-NULL"); return 0; }
    d = *desc;
    for (int i = 0; i < CATCOC_MAX_RANKS; ++i) if (!d.peers[i]) d.peers[i] = (const void *)16;
    if (make_splitk_plan(tiling, &d, 0, 0, sp)) return 0;
    ok();
    if (splitK) *splitK = sp.f;
    if (tiles) *tiles = sp.tiles;
    return sp.workspaceBytes;
}

uint32_t catcoc_get_task_count(int commType, const CocTilingParams *tiling, const CatcocSymmetricDesc *desc)
{
    Plan p;
    CatcocSymmetricDesc d;
    if (desc == nullptr || tiling == nullptr) { fail(E_NULL, "tiling and desc must be non-NULL"); return 0; }
    d = *desc;
    d.flags &= ~CATCOC_OUTBOUND_MASK;
    for (int i = 0; i < CATCOC_MAX_RANKS; ++i) if (!d.peers[i]) d.peers[i] = (const void *)16;
    const int dataType = commType == QUANT_MATMUL_REDUCE_SCATTER ? INT8 : FP16;
    if (make_plan(commType, dataType, tiling, &d, 0, 0, p)) return 0;
    ok();
    return p.args.sched.coreLoops;
}

int catcoc_task_tile(int commType, const CocTilingParams *tiling, const CatcocSymmetricDesc *desc, uint32_t task,
                     uint32_t *targetRank, uint32_t *row, uint32_t *col, uint32_t *wsRow)
{
    Plan p;
    CatcocSymmetricDesc d;
    if (desc == nullptr || tiling == nullptr) { fail(E_NULL, "tiling and desc must be non-NULL"); return 0; }
    d = *desc;
    d.flags &= ~CATCOC_OUTBOUND_MASK;
    for (int i = 0; i < CATCOC_MAX_RANKS; ++i) if (!d.peers[i]) d.peers[i] = (const void *)16;
    const int dataType = commType == QUANT_MATMUL_REDUCE_SCATTER ? INT8 : FP16;
    if (make_plan(commType, dataType, tiling, &d, 0, 0, p)) return 0;
    ok();
    TileInfo ti;
    if (!task_tile(p.args.sched, task, ti)) return 0;
    if (targetRank) *targetRank = ti.targetRank;
    if (row) *row = ti.row;
    if (col) *col = ti.col;
    if (wsRow) *wsRow = ti.wsRow;
    return 1;
}

uint32_t catcoc_task_tiles(int commType, const CocTilingParams *tiling, const CatcocSymmetricDesc *desc, uint32_t firstTask, uint32_t count,
                           uint32_t *targetRank, uint32_t *row, uint32_t *col, uint32_t *wsRow)
{
    Plan p;
    CatcocSymmetricDesc d;
    if (desc == nullptr || tiling == nullptr) { fail(E_NULL, "tiling and desc must be non-NULL"); return 0; }
    d = *desc;
    d.flags &= ~CATCOC_OUTBOUND_MASK;
    for (int i = 0; i < CATCOC_MAX_RANKS; ++i) if (!d.peers[i]) d.peers[i] = (const void *)16;
    const int dataType = commType == QUANT_MATMUL_REDUCE_SCATTER ? INT8 : FP16;
    if (make_plan(commType, dataType, tiling, &d, 0, 0, p)) return 0;   // planned once for the whole range
    ok();
    uint32_t n = 0;
    for (; n < count; ++n) {
        TileInfo ti;
        if (!task_tile(p.args.sched, firstTask + n, ti)) break;
        if (targetRank) targetRank[n] = ti.targetRank;
        if (row) row[n] = ti.row;
        if (col) col[n] = ti.col;
        if (wsRow) wsRow[n] = ti.wsRow;
    }
    return n;
}

int catcoc_launch_tile(int commType, const CocTilingParams *tiling, const CatcocSymmetricDesc *desc, uint32_t wg, uint32_t *task,
                       uint32_t *targetRank, uint32_t *row, uint32_t *col, uint32_t *wsRow)
{
    Plan p;
    CatcocSymmetricDesc d;
    if (desc == nullptr || tiling == nullptr) { fail(E_NULL, "tiling and desc must be non-NULL"); return 0; }
    d = *desc;
    d.flags &= ~CATCOC_OUTBOUND_MASK;
    for (int i = 0; i < CATCOC_MAX_RANKS; ++i) if (!d.peers[i]) d.peers[i] = (const void *)16;
    const int dataType = commType == QUANT_MATMUL_REDUCE_SCATTER ? INT8 : FP16;
    if (make_plan(commType, dataType, tiling, &d, 0, 0, p)) return 0;
    ok();
    const SchedParams &s = p.args.sched;
    const bool linear = (p.args.flags & GF_LINEAR_ORDER) != 0;
    uint32_t t;
    TileInfo ti;
    if (p.dma) {
        if (!launch_tile(s, wg, linear, p.args.keptRank, t, ti)) return 0;
    } else {
        if (wg >= s.coreLoops) return 0;
        t = launch_order_task(s, wg, linear, p.args.keptRank);
        if (!task_tile(s, t, ti)) return 0;
    }
    if (task) *task = t;
    if (targetRank) *targetRank = ti.targetRank;
    if (row) *row = ti.row;
    if (col) *col = ti.col;
    if (wsRow) *wsRow = ti.wsRow;
    return 1;
}

uint32_t catcoc_launch_task(int commType, const CocTilingParams *tiling, const CatcocSymmetricDesc *desc, uint32_t wg)
{
    Plan p;
    CatcocSymmetricDesc d;
    if (desc == nullptr || tiling == nullptr) { fail(E_NULL, "tiling and desc must be non-NULL"); return 0xffffffffu; }
    d = *desc;
    d.flags &= ~CATCOC_OUTBOUND_MASK;
    for (int i = 0; i < CATCOC_MAX_RANKS; ++i) if (!d.peers[i]) d.peers[i] = (const void *)16;
    const int dataType = commType == QUANT_MATMUL_REDUCE_SCATTER ? INT8 : FP16;
    if (make_plan(commType, dataType, tiling, &d, 0, 0, p)) return 0xffffffffu;
    ok();
    const SchedParams &s = p.args.sched;
    if (wg >= s.coreLoops) return 0xffffffffu;
    if (!p.dma) return launch_order_task(s, wg, (p.args.flags & GF_LINEAR_ORDER) != 0, p.args.keptRank);
    return launch_task(s, wg, (p.args.flags & GF_LINEAR_ORDER) != 0, p.args.keptRank);
}

// The plan of a launch that may run kept tiles as halves: on the aligned 128-row kernel, on no flexible or small tiles.
static bool plan_halves(int commType, int dataType, const CocTilingParams *tiling, const CatcocSymmetricDesc *desc, uint32_t transA, uint32_t transB, Plan &p)
{
    if (desc == nullptr || tiling == nullptr) { fail(E_NULL, "tiling and desc must be non-NULL"); return false; }
    CatcocSymmetricDesc d = *desc;
    for (int i = 0; i < CATCOC_MAX_RANKS; ++i) if (!d.peers[i]) d.peers[i] = (const void *)16;
    if (make_plan(commType, dataType, tiling, &d, transA, transB, p)) return false;
    ok();
    GemmArgs g;
    if (!p.dma || p.args.sched.m0 != 128) return false;
    if (p.preferFlex) p.args.splitK = 0;   // (as the launchers)
    return planned_small(p, !p.preferFlex, p.preferFlex, g).rows == 0 && (!p.preferFlex || keep_aligned(p.args));
}

uint32_t catcoc_kept_split_tiles(int commType, int dataType, const CocTilingParams *tiling, const CatcocSymmetricDesc *desc,
                                 uint32_t transA, uint32_t transB)
{
    Plan p;
    return plan_halves(commType, dataType, tiling, desc, transA, transB, p) ? 8u * split_kept_tiles(p.args, p.args.K * elem_size(p.dtype) / 64u) : 0u;
}

uint32_t catcoc_tail_split_tiles(int commType, int dataType, const CocTilingParams *tiling, const CatcocSymmetricDesc *desc,
                                 uint32_t transA, uint32_t transB)
{
    Plan p;
    return plan_halves(commType, dataType, tiling, desc, transA, transB, p) ? 8u * split_tail_tiles(p.args, split_kept_tiles(p.args, p.args.K * elem_size(p.dtype) / 64u)) : 0u;
}

void catcoc_last_launch(CatcocLaunchInfo *info)
{
    if (info != nullptr) *info = g_launch;
}

uint32_t catcoc_workgroup_task(uint32_t wg, uint32_t tasks, uint32_t flags)
{
    return workgroup_task(wg, tasks, (flags & CATCOC_FLAG_LINEAR_ORDER) != 0);
}

// ---- dynamic_tiling host logic ------------------------------------------------

int catcoc_check_comm_interval_reduce_scatter(const CocTilingParams *t, int rankSize, int blockNum)
{
    return rankSize > 0 && ((int64_t)blockNum * t->commInterval) % rankSize == 0;
}

static int32_t max_peer_mem_per_rank(int rankSize)
{
    // (LCAL_BUFF_BYTES - FLAG_BUFF_BYTES) / INPUT_DTYPE / rankSize / MAX_BLOCK_COUNT, info.h:24-27
    return (204 * 1024 * 1024 - 5 * 512 * 1024) / 2 / rankSize / 2;
}

int catcoc_check_comm_interval_allreduce(const CocTilingParams *t, int rankSize, int blockNum)
{
    if (rankSize <= 0) return 0;
    return t->commInterval * t->m0 * t->n0 * (uint32_t)blockNum < (uint32_t)max_peer_mem_per_rank(rankSize);
}

int catcoc_check_comm_interval_allgather(const CocTilingParams *t, int rankSize)
{
    if (rankSize <= 0) return 0;
    const uint32_t kLoop = t->k0 ? ceil_div(t->k, t->k0) : 0u;
    return t->commInterval * t->m0 * t->k0 * kLoop < (uint32_t)max_peer_mem_per_rank(rankSize);
}

int catcoc_get_tilings(const CocTilingParams *base, int commType, int rankSize, int blockNum, CocTilingParams *out, int maxOut)
{
    // search space of tiling.h:19-22 in its nesting order: interval (outer), tile M, then the split pairs
    static const uint32_t intervals[] = {4, 6, 8, 12, 14};
    static const uint32_t tileMs[] = {4, 8, 16, 32, 64};
    static const uint32_t splits[][2] = {{1, 16}, {1, 20}};
    if (base == nullptr) { fail(E_NULL, "base tiling is NULL"); return 0; }
    int n = 0;
    for (uint32_t ci : intervals)
        for (uint32_t tm : tileMs)
            for (auto &sp : splits) {
                CocTilingParams t = *base;
                t.commInterval = ci;
                t.commTileM = tm;
                t.commBlockM = tm;
                t.commNpuSplit = sp[0];
                t.commDataSplit = sp[1];
                bool valid = true;
                if (commType == ALLGATHER_MATMUL) valid = catcoc_check_comm_interval_allgather(&t, rankSize);
                else if (commType == MATMUL_REDUCE_SCATTER || commType == QUANT_MATMUL_REDUCE_SCATTER)
                    valid = catcoc_check_comm_interval_reduce_scatter(&t, rankSize, blockNum);
                else if (commType == MATMUL_ALLREDUCE) valid = catcoc_check_comm_interval_allreduce(&t, rankSize, blockNum);
                if (!valid) continue;
                if (out && n < maxOut) out[n] = t;
                ++n;
            }
    return n;
}

uint32_t catcoc_get_splitk_factor(uint32_t m, uint32_t n, uint32_t k, uint32_t coreNum, uint32_t m0, uint32_t n0, uint32_t k0)
{
    if (!m0 || !n0 || !k0 || !coreNum) return 1;
    return splitk_factor(m, n, k, coreNum, m0, n0, k0);
}

void catcoc_default_tiling(CocTilingParams *t, uint32_t m, uint32_t k, uint32_t n, uint32_t rankSize)
{
    t->m = m; t->k = k; t->n = n;
    t->m0 = 128; t->k0 = 256; t->n0 = 256;
    t->commTileM = 64;
    t->commInterval = 20;
    t->commNpuSplit = 1;
    t->commDataSplit = 2;
    t->commBlockM = 64;
    t->rankSize = rankSize;
}

// ---- schedulers on the host ---------------------------------------------------

void catcoc_swizzle_block_coord(uint32_t off, uint32_t dir, uint32_t loopsM, uint32_t loopsN, uint32_t task, uint32_t *mIdx, uint32_t *nIdx)
{
    swizzle_block_coord(off, dir, loopsM, loopsN, task, *mIdx, *nIdx);
}

void catcoc_splitk_block_coord(uint32_t off, uint32_t dir, uint32_t loopsM, uint32_t loopsN, uint32_t kTiles, uint32_t f,
                               uint32_t task, uint32_t *mIdx, uint32_t *nIdx, uint32_t *kIdx, uint32_t *slice)
{
    splitk_block_coord(off, dir, loopsM, loopsN, kTiles, f, task, *mIdx, *nIdx, *kIdx, *slice);
}

uint32_t catcoc_splitk_actual_k(uint32_t K, uint32_t k0, uint32_t f, uint32_t slice) { return splitk_actual_k(K, k0, f, slice); }

uint32_t catcoc_splitk_launch_task(uint32_t off, uint32_t dir, uint32_t loopsM, uint32_t loopsN, uint32_t f, uint32_t wg)
{
    return splitk_launch_task(off, dir, loopsM, loopsN, f, wg);
}

void catcoc_allgather_block_coord(uint32_t off, uint32_t dir, uint32_t P, uint32_t commInterval, uint32_t loopsMRank,
                                  uint32_t loopsN, uint32_t task, uint32_t *mIdx, uint32_t *nIdx)
{
    allgather_block_coord(off, dir, P, commInterval, loopsMRank, loopsN, task, *mIdx, *nIdx);
}

void catcoc_comm_block_idx(uint32_t dir, uint32_t P, uint32_t splitRow, uint32_t splitCol, uint32_t dataLoopsInRank,
                           uint32_t task, uint32_t *dataIdx, uint32_t *rankIdx)
{
    comm_block_idx(dir, P, splitRow, splitCol, dataLoopsInRank, task, *dataIdx, *rankIdx);
}

int catcoc_device_info(int *cuCount, int *clockMHz, char *name, int nameLen)
{
    int dev = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess)
        return fail(E_LAUNCH, "no HIP device");
    if (cuCount) *cuCount = prop.multiProcessorCount;
    if (clockMHz) *clockMHz = prop.clockRate / 1000;
    if (name && nameLen > 0) { strncpy(name, prop.gcnArchName, nameLen - 1); name[nameLen - 1] = 0; }
    ok();
    return 0;
}

const char *catcoc_version(void) { return "catcoc-hip 0.2 (gfx950)"; }

void catcoc_pipelined_quant_matmul_reduce_scatter(void *computeStream, void *commStream, uint64_t fftsAddr, uint8_t *x1, uint8_t *x2,
                                                  uint8_t *scale_x1, uint8_t *scale_x2, uint8_t *bias, uint8_t *c_accum, uint8_t *d_out,
                                                  uint8_t *symmetricPtr, CocTilingParams *tiling, uint32_t transA, uint32_t transB,
                                                  uint32_t outDataType, uint32_t deterministic)
{
    (void)fftsAddr;
    launch_pipelined(true, INT8, computeStream, commStream, x1, x2, scale_x1, scale_x2, bias, c_accum, d_out, symmetricPtr, tiling, transA,
                     transB, outDataType, deterministic);
}

CatcocPipelinedPlan *catcoc_pipelined_plan_create(uint32_t maxRounds)
{
    if (maxRounds == 0 || maxRounds > 65536u) { fail(E_TILING, "maxRounds %u out of range 1..65536", maxRounds); return nullptr; }
    CatcocPipelinedPlan *p = new (std::nothrow) CatcocPipelinedPlan();
    if (p == nullptr) { fail(E_LAUNCH, "out of host memory"); return nullptr; }
    if (!plan_make_events(*p, maxRounds)) { delete p; return nullptr; }
    ok();
    return p;
}

void catcoc_pipelined_plan_destroy(CatcocPipelinedPlan *plan)
{
    if (plan == nullptr) return;
    plan_destroy_events(*plan);
    delete plan;
}

uint32_t catcoc_pipelined_round_count(int commType, const CocTilingParams *tiling, const CatcocSymmetricDesc *desc)
{
    if (desc == nullptr || desc->magic != CATCOC_DESC_MAGIC) { fail(E_DESC, "desc does not point at a CatcocSymmetricDesc"); return 0; }
    if (commType != MATMUL_REDUCE_SCATTER && commType != QUANT_MATMUL_REDUCE_SCATTER) {
        fail(E_DTYPE, "the round-pipelined form exists for the reduce-scatter operators (commType %d)", commType);
        return 0;
    }
    CatcocSymmetricDesc q = *desc;
    for (int i = 0; i < CATCOC_MAX_RANKS; ++i) if (!q.peers[i]) q.peers[i] = (const void *)16;
    q.flags &= ~CATCOC_OUTBOUND_MASK;
    q.workspace = nullptr;
    q.splitK = 0;
    Plan p;
    if (make_plan(commType, commType == QUANT_MATMUL_REDUCE_SCATTER ? INT8 : FP16, tiling, &q, 0, 0, p)) return 0;
    ok();
    return ceil_div(p.args.sched.coreLoops, p.args.sched.blockPerComm);
}

void catcoc_pipelined_matmul_reduce_scatter(void *computeStream, void *commStream, int dataType, uint8_t *a, uint8_t *b, uint8_t *c,
                                            uint8_t *symmetricPtr, CocTilingParams *tiling, uint32_t transA, uint32_t transB,
                                            uint32_t deterministic)
{
    launch_pipelined(false, dataType, computeStream, commStream, a, b, nullptr, nullptr, nullptr, nullptr, c, symmetricPtr, tiling, transA,
                     transB, (uint32_t)dataType, deterministic);
}

void catcoc_reduce_add(void *stream, uint8_t *dst, uint8_t *src, uint64_t elementCount, uint32_t splitkFactor, uint32_t outDataType)
{
    if (!dst || !src) { fail(E_NULL, "dst and src must be non-NULL"); return; }
    if (splitkFactor == 0) { fail(E_TILING, "splitkFactor must be at least 1"); return; }
    if (outDataType != 0 && outDataType != FP16 && outDataType != BF16) { fail(E_DTYPE, "outDataType %u must be 0 (fp32), FP16 or BF16", outDataType); return; }
    if (elementCount == 0) { ok(); return; }
    if ((uintptr_t)src % 16 != 0 || (uintptr_t)dst % 16 != 0 || (splitkFactor > 1 && elementCount % 4 != 0)) {
        fail(E_SHAPE, "reduce-add needs 16-byte aligned buffers and, with more than one slice, an element count that is a multiple of 4");
        return;
    }
    const int e = launch_reduce_add(dst, (const float *)src, elementCount, splitkFactor, outDataType, stream);
    if (e) { fail(E_LAUNCH, "kernel launch failed: %s", hipGetErrorString((hipError_t)e)); return; }
    ok();
}

int catcoc_verify(const float *out, const float *gold, uint64_t count, int dataType, uint32_t computeTimes, uint64_t *nBad, double *meanRelErr)
{
    // examples/utils/utils.py:44-52 and verify_result.py:34-43,88-117
    if ((!out || !gold) && count) { fail(E_NULL, "out and gold must be non-NULL"); return 0; }
    if (dataType != FP16 && dataType != BF16) { fail(E_DTYPE, "dataType %d must be FP16 or BF16", dataType); return 0; }
    const float rtol = dataType == FP16 ? (computeTimes < 2048 ? 1.0f / 256 : 1.0f / 128) : (computeTimes < 2048 ? 1.0f / 128 : 1.0f / 64);
    const double meanLimit = dataType == FP16 ? 1.0 / 1024 : 1.0 / 128;
    uint64_t bad = 0;
    double sum = 0.0;
    for (uint64_t i = 0; i < count; ++i) {
        float o = out[i], g = gold[i];
        if (isnan(o) || isinf(o)) o = 0.0f;       // NaN / Inf are zeroed before the comparison
        if (isnan(g) || isinf(g)) g = 0.0f;
        const float scale = fabsf(g) > 1.0f ? fabsf(g) : 1.0f;
        const float diff = o - g;
        if (fabsf(diff) - rtol * scale > 0.0f) ++bad;
        sum += (double)(diff / scale);
    }
    const double mean = count ? fabs(sum / (double)count) : 0.0;
    if (nBad) *nBad = bad;
    if (meanRelErr) *meanRelErr = mean;
    ok();
    return bad == 0 && mean <= meanLimit;
}

void catcoc_comm_block_idx_ex(uint32_t dir, uint32_t deterministic, uint32_t P, uint32_t splitRow, uint32_t splitCol,
                              uint32_t dataLoopsInRank, uint32_t task, uint32_t *dataIdx, uint32_t *rankIdx)
{
    comm_block_idx_ex(dir, deterministic != 0, P, splitRow, splitCol, dataLoopsInRank, task, *dataIdx, *rankIdx);
}

uint32_t catcoc_comm_core_loop(uint32_t deterministic, uint32_t P, uint32_t splitRow, uint32_t splitCol, uint32_t dataLoopsInRank)
{
    return comm_core_loop(deterministic != 0, P, splitRow, splitCol, dataLoopsInRank);
}

}  // extern "C"
