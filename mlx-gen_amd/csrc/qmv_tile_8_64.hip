// qmv_tile_8_64.hip — the decode GEMV's tile kernels for Q8, group size 64.
#include "qmv_mfma.h"

namespace mlxq {
MLXQ_QMV_TILE(8, 64)
}  // namespace mlxq
