// The quantized matmul of any contraction length, tiles of 64 routes.
#include "mf_qmm_kernels.h"

namespace mf {
template hipError_t launch_qmm_tiles<kTileTokens>(hipStream_t, int, const QmmArgs&, int, uint32_t, const QmmArgs*, uint32_t, bool);
}  // namespace mf
