// Both quantized matmuls for tiles of 32 routes.
#include "mf_qmm_kernels.h"

namespace mf {
template hipError_t launch_qmm_tiles<kSmallTile>(hipStream_t, int, const QmmArgs&, int, uint32_t, const QmmArgs*, uint32_t, bool);
template hipError_t launch_kres_tiles<kSmallTile>(hipStream_t, int, const QmmArgs&, uint32_t, const QmmArgs*, uint32_t);
}  // namespace mf
