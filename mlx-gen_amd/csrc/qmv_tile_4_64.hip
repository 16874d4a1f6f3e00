// qmv_tile_4_64.hip — the decode GEMV's tile kernels for Q4, group size 64.
#include "qmv_mfma.h"

namespace mlxq {
MLXQ_QMV_TILE(4, 64)
}  // namespace mlxq
