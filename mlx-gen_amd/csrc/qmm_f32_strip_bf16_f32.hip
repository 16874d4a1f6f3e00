// qmm_f32_strip_bf16_f32.hip — the factored f32 GEMM for bf16 activations and f32 scales, and the
// dispatch over the operand mixes.
#include "qmm_f32_strip.h"

namespace mlxq {

MLXQ_STRIP_ENTRY(run_strip_bf16_f32, uint16_t, float)

// Whether a tile's rows fit 32-bit byte offsets (operands of any number of rows do).
bool qmm_f32_strip_fits(int64_t K, int64_t N) { return K % 64 == 0 && K < (1LL << 22) && N < (1LL << 22); }

int run_qmm_f32_strip(const void* x, int x_dtype, int64_t M, int64_t K, const uint32_t* wq, const void* s,
                      const void* b, int sb_dtype, int64_t N, int gs, int bits, void* y, const F32Epilogue& epi,
                      hipStream_t st) {
  if (M == 0 || N == 0) return MLXQ_OK;
  const bool sb16 = sb_dtype == MLXQ_BFLOAT16;
  if (x_dtype == MLXQ_FLOAT32)
    return sb16 ? run_strip_f32_bf16(x, M, K, wq, s, b, N, gs, bits, y, epi, st)
                : run_strip_f32_f32(x, M, K, wq, s, b, N, gs, bits, y, epi, st);
  if (x_dtype == MLXQ_FLOAT16)
    return sb16 ? run_strip_f16_bf16(x, M, K, wq, s, b, N, gs, bits, y, epi, st)
                : run_strip_f16_f32(x, M, K, wq, s, b, N, gs, bits, y, epi, st);
  return run_strip_bf16_f32(x, M, K, wq, s, b, N, gs, bits, y, epi, st);
}

}  // namespace mlxq
