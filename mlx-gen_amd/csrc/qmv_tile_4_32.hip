// qmv_tile_4_32.hip — the decode GEMV's tile kernels for Q4, group size 32.
#include "qmv_mfma.h"

namespace mlxq {
MLXQ_QMV_TILE(4, 32)
}  // namespace mlxq
