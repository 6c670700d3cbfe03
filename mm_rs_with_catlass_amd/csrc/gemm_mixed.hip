// Instantiates the mixed launches of 256x256 and 128x128 tiles.
#include "gemm_mixed.h"

namespace catcoc {
int launch_gemm_mixed(uint32_t dtype, const GemmArgs &args, void *stream)
{
    switch (dtype) {
        case DT_I8: return launch_mixed<DT_I8>(args, stream);
        case DT_F16: return launch_mixed<DT_F16>(args, stream);
        case DT_BF16: return launch_mixed<DT_BF16>(args, stream);
        default: return (int)hipErrorInvalidValue;
    }
}
}  // namespace catcoc
