// qmv_tile_8_128.hip — the decode GEMV's tile kernels for Q8, group size 128.
#include "qmv_mfma.h"

namespace mlxq {
MLXQ_QMV_TILE(8, 128)
}  // namespace mlxq
