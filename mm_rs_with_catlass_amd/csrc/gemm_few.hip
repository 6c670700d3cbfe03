// Instantiates the one-launch kernels for few small tiles.
#include "gemm_few.h"

namespace catcoc {
int launch_gemm_few(uint32_t dtype, const GemmArgs &args, int tileRows, int tileCols, void *stream)
{
    switch (dtype) {
        case DT_I8: return launch_few<DT_I8>(args, tileRows, tileCols, stream);
        case DT_F16: return launch_few<DT_F16>(args, tileRows, tileCols, stream);
        case DT_BF16: return launch_few<DT_BF16>(args, tileRows, tileCols, stream);
        default: return (int)hipErrorInvalidValue;
    }
}
}  // namespace catcoc
