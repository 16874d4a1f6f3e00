// qmm_f32_strip_f16_f32.hip — the factored f32 GEMM for f16 activations and f32 scales.
#include "qmm_f32_strip.h"

namespace mlxq {
MLXQ_STRIP_ENTRY(run_strip_f16_f32, _Float16, float)
}  // namespace mlxq
