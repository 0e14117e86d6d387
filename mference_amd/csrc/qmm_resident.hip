// The quantized matmul of contractions of up to 512, tiles of 64 routes.
#include "mf_qmm_kernels.h"

namespace mf {
template hipError_t launch_kres_tiles<kTileTokens>(hipStream_t, int, const QmmArgs&, uint32_t, const QmmArgs*, uint32_t);
}  // namespace mf
