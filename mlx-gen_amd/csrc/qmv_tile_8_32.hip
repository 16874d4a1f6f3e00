// qmv_tile_8_32.hip — the decode GEMV's tile kernels for Q8, group size 32.
#include "qmv_mfma.h"

namespace mlxq {
MLXQ_QMV_TILE(8, 32)
}  // namespace mlxq
