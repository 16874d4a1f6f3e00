// qmm_f32_strip_bf16_f32.hip — the factored f32 GEMM for bf16 activations and f32 scales, and the
// dispatch over the operand mixes.
#include "qmm_f32_strip.h"

namespace mlxq {

MLXQ_STRIP_ENTRY(run_strip_bf16_f32, uint16_t, float)

// Whether the factored kernel takes a problem: K in whole steps, a tile's rows within 32-bit byte offsets
// (operands of any number of rows are), and not f32 activations at group size 32.  There the three-pass
// kernel is the more precise one: the factored form's rounding of x is multiplied by s * c, which is
// larger than the weight s * c + b that the three-pass form multiplies it by (error against 64 bits at
// N(0, 0.02) weights, Q4 / Q8: 3.5e-6 / 3.7e-6 three-pass, 6.1e-6 factored), and x . c overflows for
// |x| from 4e34.  It is the slower one ([65, 6144] x [12288, 6144]^T 227 us against 74).  fp16 and bf16
// activations have exact products with the codes (1.4e-7 against 2.4e-6).
bool qmm_f32_strip_fits(int x_dtype, int64_t K, int64_t N, int gs) {
  return K % 64 == 0 && K < kStripReach && N < kStripReach && !(x_dtype == MLXQ_FLOAT32 && gs == 32);
}

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
