// qmm_f32_strip_f16_bf16.hip — the factored f32 GEMM for f16 activations and bf16 scales.
#include "qmm_f32_strip.h"

namespace mlxq {
MLXQ_STRIP_ENTRY(run_strip_f16_bf16, _Float16, uint16_t)
}  // namespace mlxq
