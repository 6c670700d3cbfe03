// Instantiates the one-workgroup-per-CU kernels of 128-column tiles.
#include "gemm_mid.h"

namespace catcoc {
int launch_gemm_mid(uint32_t dtype, const GemmArgs &args, int tileRows, void *stream)
{
    switch (dtype) {
        case DT_I8: return launch_mid<DT_I8>(args, tileRows, stream);
        case DT_F16: return launch_mid<DT_F16>(args, tileRows, stream);
        case DT_BF16: return launch_mid<DT_BF16>(args, tileRows, stream);
        default: return (int)hipErrorInvalidValue;
    }
}
}  // namespace catcoc
