// qmm_f32_strip_f32_f32.hip — the factored f32 GEMM for f32 activations and f32 scales.
#include "qmm_f32_strip.h"

namespace mlxq {
MLXQ_STRIP_ENTRY(run_strip_f32_f32, float, float)
}  // namespace mlxq
