// 256x256 tiles and, in the same launch, small ones: large problems whose tiles do not come out even.
//
// The large tile is the one with the fewest bytes per product (gemm_dma_kernel.h, 256 rows on eight waves) in flexible mode: rows past
// a rank's end, columns and bytes of k past the last one are nobody's business.  With one workgroup per CU a launch lasts as many rounds
// as its fullest CU, and a last round of a few tiles takes nearly as long as a full one; and a reduce-scatter's kept rows, in a few large
// tiles, would wait for the peers' stream through as many CUs.  So some rows run on 128x128 tiles (gemm_mid.h) in the same launch: the
// kept ones and as many more as shorten the launch by its estimate (mixed_rows).  The large tiles start first.
//
// Bound by the matrix pipes at their power limit: a large tile takes 5 + 1.1 us per 128 bytes of k where some CUs are idle, 1.5 per 128 bytes where none is
// (1.45 PFLOP/s in 16 bits), a small one 5 + 0.37 and 0.46.  Time per call, calls behind each other and their
// operands out of HBM, 128-row tiles -> this, reduce-scatters with stored tiles, as [n,k]: fp16 8144x5120x1696 of eight ranks (7126 rows on
// 196 large tiles, the kept 1018 on 112 small ones beside them) 184 -> 168 us (162.5 on 16x16 MFMAs), W8A8 2680x3200x6912 124 -> 81, 1384x6080x7936 145 -> 85,
// 3824x5632x6400 217 -> 157, bf16 4236x4952x3904 of four 284 -> 196.  Which launches: small_tile().
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemm_mid.h"

namespace catcoc {

template <uint32_t DT, bool TB>
__global__ void __launch_bounds__(512, 1) gemm_mixed_kernel(const GemmArgs args)
{
    __shared__ __attribute__((aligned(1024))) unsigned char smem[FLEX_POOL8];
    static_assert(MidGeom<4>::POOL <= FLEX_POOL8, "the small tiles fit");
    const FlexParams &f = args.fx;
    if (blockIdx.x < f.largeTiles) {
        dma_tile<DT, 4, TB, false, false, false, 2, 3, false, false, false, 1>(args, smem, blockIdx.x, 0, 1u, 0);
    } else {
        mid_tile<DT, TB, 4, DT != DT_I8>(args, smem, blockIdx.x - f.largeTiles, ceil_div(f.holeRows, 128u), ceil_div(args.N, 128u), f.hole0, f.hole0 + f.holeRows);
    }
}

template <uint32_t DT>
inline int launch_mixed(const GemmArgs &args, void *stream)
{
    const dim3 grid(args.fx.largeTiles + ceil_div(args.fx.holeRows, 128u) * ceil_div(args.N, 128u)), block(512);
    if (args.transB) hipLaunchKernelGGL((gemm_mixed_kernel<DT, true>), grid, block, 0, (hipStream_t)stream, args);
    else hipLaunchKernelGGL((gemm_mixed_kernel<DT, false>), grid, block, 0, (hipStream_t)stream, args);
    return (int)hipGetLastError();
}

}  // namespace catcoc
