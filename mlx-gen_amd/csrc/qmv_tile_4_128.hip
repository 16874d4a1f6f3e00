// qmv_tile_4_128.hip — the decode GEMV's tile kernels for Q4, group size 128.
#include "qmv_mfma.h"

namespace mlxq {
MLXQ_QMV_TILE(4, 128)
}  // namespace mlxq
