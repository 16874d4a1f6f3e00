// qmm_f32_strip.h — the large-M quantized GEMM in f32 (y[M,N] = x[M,K] . W^T, K % 64 == 0) for the
// operand mixes MLX computes in f32: fp16 or f32 activations, and bf16 ones against f32 scales.
//
// Since
//     x . w = sum_g ( s_g * sum_{k in g} x_k c_k  +  b_g * X_g ),   X_g = sum_{k in g} x_k,
// the codes c (integers below 256, exact in bf16 and fp16) are one MFMA operand and the activations
// the other, with no dequantization: fp16 and bf16 activations as they are (one pass, every product
// exact), f32 ones as two bf16 values whose sum holds them to 16 significant bits (two passes,
// v_hi = bf16(v), v_lo = bf16(v - v_hi)).  Each group's product accumulates in `acc`, whose first
// MFMA starts from zero, and is folded into the running sum by one FMA per output, y += s_g * acc.
// The bias term runs on the f32 matrix cores, two groups per MFMA, between the two groups' folds.
// s_g * acc and b_g * X_g are large and of opposite sign, so how many groups have only one of them in
// the running sum sets the error: [4096, 1280] fp16 x Q4 was 2.1e-7 off the 64-bit product with 16
// groups per bf16 MFMA (X in three bf16 terms), 1.7e-7 with four, 1.6e-7 with two after both folds,
// and is 1.4e-7 in this form, as with two FMAs per output and group.
//
// Workgroup: 8 waves, tile BM (128 or 64) x 256 TN, K advanced 64 per step; wave w owns TN strips of 32
// columns, all BM rows of them.  Small grids (strip_shape) take KS = 2 or 4 K-groups of 8 / KS
// waves instead: each group walks its own share of K, with its own activation ring, over the same
// 256 / KS columns, and the partial sums meet in LDS at the end.  No unit is
// saturated; what bounds it is how far a SIMD's two waves overlap the matrix work with the vector work
// (code conversions, folds), which takes about as long (counters, share of the SIMDs' cycles, matrix /
// vector at 4 cycles an instruction, and of the CUs' cycles, LDS at 8 cycles a KB: [4096, 1280] fp16 x Q4
// [10240, 1280]^T 37 / 44 / 41 %, [4608, 3072] f32 x Q4 [12288, 3072]^T 53 / 46 / 31 %).  Trading LDS
// reads for conversions moves it by less than 10 % either way (strip_tile).
// The weights never pass through LDS: a lane loads its own column's packed words two steps ahead and
// converts them straight into its MFMA operand, each code once per workgroup, and with the codes
// as the MFMA's B side a lane holds 16 rows of ONE column, so the fold's scale is a single register.
// fp16 and bf16 activations go global -> LDS by direct-to-LDS loads three steps ahead into a 4-stage
// ring; f32 ones through registers, where they are split and summed, one step ahead.
// The fold of a group is interleaved with the next group's first MFMAs block by block, so the vector
// work of one block runs under the MFMAs of the others.
//
// Same-process A/B against the kernel it replaces (128 x 256 tiles of 64 x 64 per wave, codes and
// split activations through LDS, fp16 split into two bf16 passes; LoRA in a launch of its own):
// [4096, 1280] fp16 x Q4 [10240, 1280]^T with bias 281 -> 154 us; [77, 1280] fp16 x Q8 [5120, 1280]^T
// with bias and GELU 50.5 -> 8.7 (21.0 without K-groups); [4608, 3072] f32 x Q4 [12288, 3072]^T with bias, rank-32 LoRA and
// GELU 1043 -> 795.
//
// All buffer resources start at the tile's own first row, so 32-bit offsets reach any operand, and
// rows past M or N read as zero.
#pragma once

#include <type_traits>

#include "mlxq_common.h"

namespace mlxq {

namespace {

constexpr int kStripGroupM = 8;  // M-tiles per group of the tile order
constexpr int kStripFlags = 0x00020000;  // raw buffer resource word 3 for gfx9-family loads
// Widths (K and N) below which the rows of a 64-row tile stay below 2^31 bytes, as do those of a 128-row
// tile below half of it.
constexpr int64_t kStripReach = 1LL << 23;
// Added to an activation offset (below 2^31), past the tile's rows: zero.
constexpr uint32_t kStripPast = 0x80000000u;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// Consecutive workgroup ids are spread over the 8 XCDs, so each XCD is given a contiguous slice of
// an order that walks groups of 8 M-tiles by all N-tiles, M fastest: the workgroups in flight on
// an XCD share weight and activation panels in its L2.
__device__ __forceinline__ void strip_coords(int64_t bid, int64_t tiles_m, int64_t tiles_n, int64_t& tm, int64_t& tn) {
  const int64_t T = tiles_m * tiles_n, per = T / 8;
  const int64_t L = bid < per * 8 ? (bid % 8) * per + bid / 8 : bid;
  const int64_t span = kStripGroupM * tiles_n;
  const int64_t g = L / span, gm0 = g * kStripGroupM;
  const int64_t gsz = tiles_m - gm0 < kStripGroupM ? tiles_m - gm0 : kStripGroupM;
  const int64_t idx = L - g * span;
  tm = gm0 + idx % gsz;
  tn = idx / gsz;
}

// Workgroup barrier that waits for this wave's LDS operations only (a release fence would also wait
// for every direct-to-LDS load in flight; the loop waits for exactly those it needs).
__device__ __forceinline__ void strip_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// A copy the compiler cannot elide: the word taken from a ring register must not share the register
// the next load in flight writes.
__device__ __forceinline__ uint32_t take(uint32_t v) {
  uint32_t r;
  asm volatile("v_mov_b32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}

// Eight codes as exact fp16 or bf16 values in code order: word kk of w (Q4), words 2kk, 2kk+1 (Q8).
// Q4: the nibbles become bytes in code order, and a byte c <= 15 read as OCP fp8 E4M3 is c * 2^-9, so
// one scaled convert makes two exact values (9 VALU ops).  Q8 to fp16: bytes under 0x64 are 1024 + c.
template <int BITS, bool F16>
__device__ __forceinline__ u32x4 codes8(const uint32_t* w, int kk) {
  u32x4 o;
  if constexpr (BITS == 4) {
    const uint32_t v = w[kk], ev = v & 0x0f0f0f0fu, od = (v >> 4) & 0x0f0f0f0fu;
    const uint32_t n0 = __builtin_amdgcn_perm(od, ev, 0x05010400u), n1 = __builtin_amdgcn_perm(od, ev, 0x07030602u);
    if constexpr (F16) {
      o[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(n0, 512.0f, false));
      o[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(n0, 512.0f, true));
      o[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(n1, 512.0f, false));
      o[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(n1, 512.0f, true));
    } else {
      o[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(n0, 512.0f, false));
      o[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(n0, 512.0f, true));
      o[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(n1, 512.0f, false));
      o[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(n1, 512.0f, true));
    }
  } else {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t v = w[2 * kk + h];
      if constexpr (F16) {
        const f16x2 k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
        const f16x2 a = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, v, 0x04010400u)) - k1024;
        const f16x2 b = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, v, 0x04030402u)) - k1024;
        o[2 * h] = __builtin_bit_cast(uint32_t, a);
        o[2 * h + 1] = __builtin_bit_cast(uint32_t, b);
      } else {
        o[2 * h] = pack_bf16x2(ubyte<0>(v), ubyte<1>(v));
        o[2 * h + 1] = pack_bf16x2(ubyte<2>(v), ubyte<3>(v));
      }
    }
  }
  return o;
}

// sum + the low (0) or high (1) fp16 half of w, in one instruction.
template <int H>
__device__ __forceinline__ float add_f16(uint32_t w, float sum) {
  if constexpr (H == 0) asm("v_fma_mix_f32 %0, %1, 1.0, %0 op_sel_hi:[1,0,0]" : "+v"(sum) : "v"(w));
  else asm("v_fma_mix_f32 %0, %1, 1.0, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(sum) : "v"(w));
  return sum;
}

}  // namespace

// XT: activation storage (float, _Float16, or uint16_t bf16 bits); SB: scale/bias storage.
template <typename XT, typename SB, int BITS, int GS, int BM, int KS, int TN>
__global__ __launch_bounds__(512) void qmm_f32_strip_kernel(const XT* __restrict__ x, int64_t M, int64_t K,
                                                            const uint32_t* __restrict__ wq,
                                                            const SB* __restrict__ scales,
                                                            const SB* __restrict__ biases, int64_t N,
                                                            float* __restrict__ y, F32Epilogue epi) {
  constexpr bool F16 = std::is_same<XT, _Float16>::value;
  constexpr bool XF32 = std::is_same<XT, float>::value;
  constexpr bool SBF = std::is_same<SB, float>::value;
  constexpr int P = XF32 ? 2 : 1;             // passes: activation parts in LDS
  constexpr int TM = BM / 32;                 // 32-row blocks per wave
  constexpr int PART = BM * 128;              // bytes of one part of one stage (BM rows of 64 values)
  constexpr int STAGE = P * PART;
  constexpr int GPB = 16;                     // groups per scale / bias table
  constexpr int SPB = GPB * GS / 64;          // K steps per table
  constexpr int SPP = SPB / 8;                // K steps per pair of groups
  constexpr int STAGES = XF32 ? 3 : 4;        // activation ring
  constexpr int NS = 8 / KS;                  // waves per K-group, TN 32-column strips each
  constexpr int BN = 32 * TN * NS;
  static_assert(KS == 1 || TN == 1, "K-groups add up one strip per wave");
  constexpr int A_ROWS = 8 * NS;              // rows one round of a K-group's loads covers
  constexpr int A_LD = BM / A_ROWS;           // 8-value chunks per thread (f32), or direct-to-LDS rounds
  static_assert(A_LD >= 1, "tile too low for the K-group");
  constexpr int NW = GS == 32 ? 2 : BITS / 4; // weight loads per lane per step (8 or 16 bytes)
  constexpr int OFF_X = STAGES * STAGE;       // per K-group: its ring, then [group % 8][BM rows] f32 sums
  constexpr int REGION = OFF_X + 8 * BM * 4;
  constexpr int OFF_S = KS * REGION;
  constexpr int SW = 32 * GPB * (int)sizeof(SB);  // per wave: [half][32 columns][8 groups] scales, then biases
  constexpr int PARTS = KS > 1 ? 8 * TM * 4096 : 0;  // the partial sums, over everything else
  constexpr int TABLES = 8 * TN * 2 * SW;
  __shared__ __attribute__((aligned(16))) unsigned char lds_all[OFF_S + TABLES > PARTS ? OFF_S + TABLES : PARTS];

  const int lane = threadIdx.x & 63, r32 = lane & 31, half = lane >> 5;
  const int wave_all = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int kg = wave_all / NS, wave = wave_all % NS, tid = threadIdx.x % (64 * NS);  // K-group; within it
  unsigned char* const lds = lds_all + kg * REGION;
  auto stage_at = [&](int t) { return lds + (XF32 ? t % 3 : t & 3) * STAGE; };
  const int64_t tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  int64_t tm, tn;
  strip_coords(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int64_t bm0 = tm * BM, bn0 = tn * BN;
  const int rows_m = (int)(M - bm0 < BM ? M - bm0 : BM), rows_n = (int)(N - bn0 < BN ? N - bn0 : BN);
  const uint32_t kwords = (uint32_t)(K * BITS / 32);
  const int groups_all = (int)(K / GS);
  // This K-group's steps [t0, t0 + T), whole groups; every group runs T_run steps, the ones past its own
  // on zero activations with zero scales (with the last step's activations, an infinity among them would
  // fold as 0 * inf).
  constexpr int UNIT = GS == 128 ? 2 : 1;  // steps
  const int units = (int)(K / (64 * UNIT));
  const int t0 = UNIT * (kg * units / KS), T = UNIT * ((kg + 1) * units / KS) - t0;
  const int T_run = UNIT * ((units + KS - 1) / KS);
  const int groups = T * 64 / GS, g_base = t0 * 64 / GS;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<XT*>(x + bm0 * K), (short)0, (int)(uint32_t)(rows_m * K * (int64_t)sizeof(XT)), kStripFlags);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint32_t*>(wq + bn0 * kwords), (short)0, (int)(uint32_t)(rows_n * (int64_t)kwords * 4), kStripFlags);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<SB*>(scales + bn0 * groups_all), (short)0, (int)(uint32_t)(rows_n * (int64_t)groups_all * (int64_t)sizeof(SB)), kStripFlags);
  const __amdgpu_buffer_rsrc_t rz = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<SB*>(biases + bn0 * groups_all), (short)0, (int)(uint32_t)(rows_n * (int64_t)groups_all * (int64_t)sizeof(SB)), kStripFlags);

  // ---- activations.  16-byte chunk c (8 values) of row r sits at chunk c ^ swz_f(r) of its row.
  // fp16 / bf16: round i of wave w fills rows A_ROWS i + 8 w .. + 7, lane L the chunk that belongs at
  // position L & 7 of row A_ROWS i + 8 w + (L >> 3).  f32: thread t loads chunk t & 7 (32 bytes) of
  // rows t / 8 + A_ROWS i.
  uint32_t x_off[A_LD];
#pragma unroll
  for (int i = 0; i < A_LD; ++i) {
    if constexpr (XF32) {
      x_off[i] = (uint32_t)(((tid >> 3) + A_ROWS * i) * K * 4 + t0 * 256 + (tid & 7) * 32);
    } else {
      const int r = A_ROWS * i + 8 * wave + (lane >> 3);
      x_off[i] = (uint32_t)((r * K + t0 * 64 + ((lane & 7) ^ swz_f(r)) * 8) * 2);
    }
  }
  auto dma_x = [&](int t) {  // !XF32
#if defined(__HIP_DEVICE_COMPILE__)
    unsigned char* const base = stage_at(t);
    const uint32_t at = t < T ? (uint32_t)t * 128u : kStripPast;
#pragma unroll
    for (int i = 0; i < A_LD; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (__attribute__((address_space(3))) void*)(base + (A_ROWS * i + 8 * wave) * 128),
                                               16, x_off[i] + at, 0, 0, 0);
#else
    (void)t;
#endif
  };
  u32x4 xr[XF32 ? A_LD : 1][2];
  auto load_x = [&](int t) {  // XF32
    const uint32_t at = t < T ? (uint32_t)t * 256u : kStripPast;
#pragma unroll
    for (int i = 0; i < A_LD; ++i)
#pragma unroll
      for (int q = 0; q < 2; ++q)
        xr[i][q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, x_off[i] + at + 16u * q, 0, 0));
  };
  float* const xtab = reinterpret_cast<float*>(lds + OFF_X);
  float xrun[XF32 ? A_LD : 1];  // GS 128: a row's sum over its group's first step
  // X of group g for tile row `row`; the lanes that share a row write the same value.
  auto put_x = [&](int row, int g, float v) { xtab[(g & 7) * BM + row] = v; };
  // f32: split step t's registers into its stage and leave the group sums.  POS: t's position in its
  // 128-wide group.
  auto stage_x = [&](int t, auto POS) {
    unsigned char* const base = stage_at(t);
#pragma unroll
    for (int i = 0; i < A_LD; ++i) {
      const int row = (tid >> 3) + A_ROWS * i, c = tid & 7;
      u32x4 hi, lo;
      float sum = 0.0f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v0 = __uint_as_float(xr[i][e >> 1][2 * (e & 1)]), v1 = __uint_as_float(xr[i][e >> 1][2 * (e & 1) + 1]);
        sum += v0 + v1;
        hi[e] = pack_bf16x2(v0, v1);
        lo[e] = pack_bf16x2(v0 - __uint_as_float(hi[e] << 16), v1 - __uint_as_float(hi[e] & 0xffff0000u));
      }
      unsigned char* const p = base + row * 128 + ((c ^ swz_f(row)) << 4);
      *reinterpret_cast<u32x4*>(p) = hi;
      *reinterpret_cast<u32x4*>(p + PART) = lo;
      // the row's 8 chunks sit in 8 consecutive lanes
      sum += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sum), 0xb1, 0xf, 0xf, true));
      sum += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sum), 0x4e, 0xf, 0xf, true));
      if constexpr (GS == 32) {
        put_x(row, 2 * t + (c >> 2), sum);
      } else {
        sum += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sum), 0x141, 0xf, 0xf, true));
        if constexpr (GS == 64) {
          put_x(row, t, sum);
        } else if constexpr (decltype(POS)::value == 0) {
          xrun[i] = sum;
        } else {
          put_x(row, t >> 1, xrun[i] + sum);
        }
      }
    }
  };
  // fp16 / bf16: the group sums of step t from its landed stage, BM / NS rows per wave, four lanes a
  // row (two chunks each).
  auto sum_x = [&](int t, auto POS) {
    constexpr int RW = BM / NS;
    static_assert(RW == 16 || RW == 8, "rows of a wave: all its lanes, or twice over");
    const int row = wave * RW + ((lane >> 2) & (RW - 1)), q = lane & 3;
    const unsigned char* const base = stage_at(t) + row * 128;
    float part[2] = {0.0f, 0.0f};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(base + (((2 * q + h) ^ swz_f(row)) << 4));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (F16) {
          part[0] = add_f16<0>(v[e], part[0]);
          part[1] = add_f16<1>(v[e], part[1]);
        } else {
          part[0] += __uint_as_float(v[e] << 16);
          part[1] += __uint_as_float(v[e] & 0xffff0000u);
        }
      }
    }
    // Every lane of a row ends with the same sum and writes it: no branch.
    float sum = part[0] + part[1];
    sum += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sum), 0xb1, 0xf, 0xf, true));
    if constexpr (GS == 32) {
      put_x(row, 2 * t + (q >> 1), sum);
    } else {
      sum += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sum), 0x4e, 0xf, 0xf, true));
      if constexpr (GS == 64) put_x(row, t, sum);
      else if constexpr (decltype(POS)::value == 0) xrun[0] = sum;
      else put_x(row, t >> 1, xrun[0] + sum);
    }
  };

  // ---- weights: column n = 32 w + r32 of the tile.  Lane half h covers, for MFMA kk of a step, 16-byte
  // chunk 4 h + kk of k (group 64 and 128), or 4 (kk >> 1) + 2 h + (kk & 1) (group 32, so that MFMAs 0, 1
  // and 2, 3 stay inside one group): its packed words are contiguous, one or two loads.
  uint32_t ncol[TN], w_off[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    ncol[j] = (uint32_t)(32 * (TN * wave + j) + r32);
    w_off[j] = (ncol[j] * kwords + (uint32_t)t0 * (2 * BITS) + (uint32_t)half * (GS == 32 ? BITS / 2 : BITS)) * 4u;
  }
  auto chunk_of = [&](int kk) { return GS == 32 ? 4 * (kk >> 1) + 2 * half + (kk & 1) : 4 * half + kk; };
  uint32_t wr[2][TN][BITS], wc[TN][BITS];
  auto load_w = [&](int t, auto SLOT) {
    constexpr int sl = decltype(SLOT)::value;
    constexpr int EACH = BITS / NW;  // words per load
#pragma unroll
    for (int jq = 0; jq < TN * NW; ++jq) {
      const int j = jq / NW, q = jq % NW;
      const uint32_t o = w_off[j] + (uint32_t)(t < T ? t : T - 1) * (8u * BITS) + (GS == 32 ? 4u * BITS * q : 16u * q);
      if constexpr (EACH == 2) {
        const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rw, o, 0, 0));
#pragma unroll
        for (int e = 0; e < 2; ++e) wr[sl][j][2 * q + e] = v[e];
      } else {
        const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, o, 0, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) wr[sl][j][4 * q + e] = v[e];
      }
    }
  };
  auto take_w = [&](auto SLOT) {
    constexpr int sl = decltype(SLOT)::value;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < BITS; ++e) wc[j][e] = take(wr[sl][j][e]);
  };

  // ---- scales and biases, 16 groups at a time: lane (h, r32) loads groups 16 b + 8 h .. + 7 of its
  // column into the wave's LDS tables, from which each group's scale and bias are read back.  Groups
  // past the last are zero.
  struct Batch { uint32_t s[SBF ? 8 : 4], z[SBF ? 8 : 4]; };
  auto load_batch = [&](int b, int j, Batch& d) {
    const int g0 = 16 * b + 8 * half;
    const uint32_t first = ncol[j] * (uint32_t)groups_all + (uint32_t)(g_base + g0), at = first * (uint32_t)sizeof(SB);
    if (16 * b + 16 <= groups && (SBF || ((groups_all | g_base) & 1) == 0)) {  // whole and dword-aligned
#pragma unroll
      for (int q = 0; q < (SBF ? 2 : 1); ++q) {
        const u32x4 s = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, at + 16u * q, 0, 0));
        const u32x4 z = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rz, at + 16u * q, 0, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          d.s[4 * q + e] = s[e];
          d.z[4 * q + e] = z[e];
        }
      }
    } else {
      uint32_t s[8], z[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t idx = g0 + e < groups ? first + (uint32_t)e : 0xffffffffu / (uint32_t)sizeof(SB);
        s[e] = load_sb_bits<SB>(rs, idx);  // past the resource: zero
        z[e] = load_sb_bits<SB>(rz, idx);
      }
#pragma unroll
      for (int e = 0; e < (SBF ? 8 : 4); ++e) {
        d.s[e] = SBF ? s[e] : (s[2 * e] & 0xffffu) | (s[2 * e + 1] << 16);
        d.z[e] = SBF ? z[e] : (z[2 * e] & 0xffffu) | (z[2 * e + 1] << 16);
      }
    }
  };
  unsigned char* const stab = lds_all + OFF_S + wave_all * TN * 2 * SW;  // [strip][scales, biases]
  auto put_tables = [&](int j, const Batch& d) {
    unsigned char* const p = stab + j * 2 * SW + half * (SW / 2) + r32 * (8 * (int)sizeof(SB));
#pragma unroll
    for (int q = 0; q < (SBF ? 2 : 1); ++q) {
      *reinterpret_cast<u32x4*>(p + 16 * q) = u32x4{d.s[4 * q], d.s[4 * q + 1], d.s[4 * q + 2], d.s[4 * q + 3]};
      *reinterpret_cast<u32x4*>(p + SW + 16 * q) = u32x4{d.z[4 * q], d.z[4 * q + 1], d.z[4 * q + 2], d.z[4 * q + 3]};
    }
  };
  auto scale_of = [&](int j, int g) {
    return SBLoad<SB>::ld(reinterpret_cast<const SB*>(stab + j * 2 * SW + ((g >> 3) & 1) * (SW / 2)) + r32 * 8, g & 7);
  };

  f32x16 acc[TM][TN], yv[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        acc[i][j][v] = 0.0f;
        yv[i][j][v] = 0.0f;
      }
  // y += b . X over the groups 2 p and 2 p + 1; this half's operands are those of group 2 p + half.
  auto bias_pair = [&](int p) {
    const int g = 2 * p + half;
    float z[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j)
      z[j] = SBLoad<SB>::ld(reinterpret_cast<const SB*>(stab + j * 2 * SW + SW + ((p >> 2) & 1) * (SW / 2)) + r32 * 8,
                            2 * (p & 3) + half);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const float xg = xtab[(g & 7) * BM + 32 * i + r32];
#pragma unroll
      for (int j = 0; j < TN; ++j)
        yv[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(g < groups ? xg : 0.0f, z[j], yv[i][j], 0, 0, 0);
    }
  };

  // ---- the loop.  Sub-step u = kk * P + part of a step multiplies fragments of one activation part
  // by the codes of MFMA kk; its fragments were read one sub-step earlier.
  constexpr int NSUB = 4 * P;
  u32x4 af[2][TM], cf[2][TN];
  int a_off[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) a_off[kk] = r32 * 128 + ((chunk_of(kk) ^ swz_f(r32)) << 4);
  auto read_a = [&](int slot, const unsigned char* base, int u) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
      af[slot][i] = *reinterpret_cast<const u32x4*>(base + (u % P) * PART + i * 4096 + a_off[u / P]);
  };
  auto convert = [&](int slot, int kk) {
#pragma unroll
    for (int j = 0; j < TN; ++j) cf[slot][j] = codes8<BITS, F16>(wc[j], kk);
  };
  float s_prev[TN] = {}, s_next[2][TN] = {};
  auto mfma = [&](const u32x4& a, const u32x4& c, const f32x16& d) {
    if constexpr (F16)
      return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, c), d, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, c), d, 0, 0, 0);
  };
  // Sub-step U (position POS of the step in a 128-wide group): a group's first sub-step folds the
  // group before, block by block, and starts its own sums from zero.
  auto sub = [&](auto U, auto POS) {
    constexpr int u = decltype(U)::value, kk = u / P;
    constexpr bool start = u % P == 0 && (GS == 32 ? kk % 2 == 0 : GS == 64 ? kk == 0 : kk == 0 && decltype(POS)::value == 0);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (start) {
#pragma unroll
        for (int v = 0; v < 16; ++v) yv[i][j][v] = fmaf(s_prev[j], acc[i][j][v], yv[i][j][v]);
        // Pinned here (else the folds sink to where y is next read), and vector and matrix instructions
        // stay on their side, so a block's old sums die before its new ones are born.
        asm volatile("" : "+v"(yv[i][j]));
        __builtin_amdgcn_sched_barrier(0x4 | 0x10 | 0x80);
        acc[i][j] = mfma(af[u & 1][i], cf[kk & 1][j], f32x16{});
      } else {
        acc[i][j] = mfma(af[u & 1][i], cf[kk & 1][j], acc[i][j]);
      }
    }
    if constexpr (start) {
#pragma unroll
      for (int j = 0; j < TN; ++j) s_prev[j] = s_next[GS == 32 ? kk / 2 : 0][j];
    }
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  Batch nb[TN];
  auto load_batches = [&](int b) {
#pragma unroll
    for (int j = 0; j < TN; ++j) load_batch(b, j, nb[j]);
  };
  // Step t: before its middle barrier the first half of its sub-steps, and (f32) the staging of step
  // t + 1; after it the loads of later steps, the rest, and the first fragments of step t + 1.
  auto step = [&](int t, auto PAR) __attribute__((always_inline)) {
    using NPAR = std::integral_constant<int, 1 - decltype(PAR)::value>;
    const unsigned char* const As = stage_at(t);
    const unsigned char* const An = stage_at(t + 1);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (GS == 32) {
        s_next[0][j] = scale_of(j, 2 * t);
        s_next[1][j] = scale_of(j, 2 * t + 1);
      } else if constexpr (GS == 64 || decltype(PAR)::value == 0) {
        s_next[0][j] = scale_of(j, GS == 64 ? t : t >> 1);
      }
    }
    if constexpr (XF32) stage_x(t + 1, NPAR{});
    auto half1 = [&](auto U) {
      constexpr int u = decltype(U)::value;
      read_a((u + 1) & 1, As, u + 1);
      if constexpr ((u + 1) % P == 0) convert(((u + 1) / P) & 1, (u + 1) / P);
      sub(U, PAR);
    };
    half1(std::integral_constant<int, 0>{});
    half1(std::integral_constant<int, 1>{});
    if constexpr (P == 2) {
      half1(std::integral_constant<int, 2>{});
      half1(std::integral_constant<int, 3>{});
    }
    // x(t + 1) was issued in step t - 2, whatever its order against w(t + 1); x(t + 2) and w(t + 2) in
    // step t - 1.
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!XF32) mlxq_vmcnt<TN * NW + A_LD>();
    strip_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (XF32) load_x(t + 2);
    else dma_x(t + 3);
    half1(std::integral_constant<int, 2 * P>{});
    if constexpr (P == 2) half1(std::integral_constant<int, 5>{});
    if constexpr (P == 2) half1(std::integral_constant<int, 6>{});
    if constexpr (!XF32) sum_x(t + 1, NPAR{});
    take_w(NPAR{});
    load_w(t + 3, NPAR{});
    read_a(0, An, 0);
    convert(0, 0);
    sub(std::integral_constant<int, NSUB - 1>{}, PAR);
    __builtin_amdgcn_sched_barrier(0);
    // A pair of groups ends with this step: their X sums were left during the step before, so all are
    // visible since the barrier, and the second group is folded in the step after.
    if (SPP == 1 || decltype(PAR)::value == 1) {
      if ((t + 1) % SPP == 0) bias_pair(t / SPP);
      if ((t + 1) % SPB == 0) {
#pragma unroll
        for (int j = 0; j < TN; ++j) put_tables(j, nb[j]);
        load_batches((t + 1) / SPB + 1);
      }
    }
  };

  // ---- prologue: batch 0's scales, x and w of the first steps (issued x(0) w(0) x(1) w(1) x(2) w(2)).
  load_batches(0);
  if constexpr (XF32) load_x(0);
  else dma_x(0);
  load_w(0, I0{});
  if constexpr (!XF32) dma_x(1);
  load_w(1, I1{});
  if constexpr (!XF32) dma_x(2);
#pragma unroll
  for (int j = 0; j < TN; ++j) put_tables(j, nb[j]);
  if constexpr (XF32) {
    stage_x(0, I0{});
    load_x(1);
  }
  take_w(I0{});
  load_batches(1);
  load_w(2, I0{});
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (!XF32) mlxq_vmcnt<TN * NW + 2 * A_LD>();  // x(0) is older than w(1), x(1), x(2) and w(2)
  strip_barrier();
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (!XF32) sum_x(0, I0{});
  read_a(0, lds, 0);
  convert(0, 0);
  int t = 0;
  for (; t + 1 < T_run; t += 2) {
    step(t, I0{});
    step(t + 1, I1{});
  }
  if (t < T_run) step(t, I0{});
  // The last pair's bias term when its second group does not exist, and the last group's fold.
  if (T_run % SPP != 0) bias_pair((T_run - 1) / SPP);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) yv[i][j][v] = fmaf(s_prev[j], acc[i][j][v], yv[i][j][v]);
  mlxq_vmcnt<0>();  // no direct-to-LDS load outlives the loop

  // ---- K-groups: every wave leaves its partial sums in LDS (over the rings and tables, which all waves
  // are past), and takes 1 / KS of its strip's 4-row pieces (i, q) to add up, in K-group order, and finish.
  constexpr int MINE = TM * 4 / KS;
  auto part = reinterpret_cast<f32x4 (*)[TM * 4][64]>(lds_all);
  if constexpr (KS > 1) {
    strip_barrier();
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        part[wave_all][4 * i + q][lane] = f32x4{yv[i][0][4 * q], yv[i][0][4 * q + 1], yv[i][0][4 * q + 2], yv[i][0][4 * q + 3]};
    strip_barrier();
  }

  // ---- epilogue: lane holds column n and rows m = 32 i + 8 q + 4 half + e: y + bias in f32, the LoRA
  // residual (xa . lbt^T on the f32 matrix cores) times its scale, the activation.
  const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(
      y + bm0 * N, (short)0, (int)(uint32_t)(rows_m * N * 4), kStripFlags);
  // (All blocks' residuals at once, in the registers of acc, made the loop itself spill: 785 -> 953 us.)
  auto finish = [&](auto ACT) {
#pragma unroll
    for (int ji = 0; ji < TN * TM; ++ji) {
      const int j = ji / TM, i = ji % TM;
      const bool n_ok = (int)ncol[j] < rows_n;
      const int64_t n = bn0 + (n_ok ? (int)ncol[j] : 0);
      const float bv = epi.bias == nullptr ? -0.0f
                       : epi.bias_bf16 ? bf16_bits_to_f32(static_cast<const uint16_t*>(epi.bias)[n])
                                       : static_cast<const float*>(epi.bias)[n];
      f32x16 r = {};
      if (epi.R > 0) {
        const int mr = 32 * i + r32 < rows_m ? 32 * i + r32 : rows_m - 1;
        for (int k = 0; k < epi.R; k += 16) {
          const f32x4* const xp = reinterpret_cast<const f32x4*>(epi.xa + (bm0 + mr) * epi.R + k + 8 * half);
          const f32x4* const lp = reinterpret_cast<const f32x4*>(epi.lbt + n * epi.R + k + 8 * half);
          const f32x4 x0 = xp[0], x1 = xp[1], l0 = lp[0], l1 = lp[1];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            r = __builtin_amdgcn_mfma_f32_32x32x2f32(x0[e], l0[e], r, 0, 0, 0);
            r = __builtin_amdgcn_mfma_f32_32x32x2f32(x1[e], l1[e], r, 0, 0, 0);
          }
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (KS > 1 && (4 * i + q) / MINE != kg) continue;  // wave-uniform
        f32x4 o;
        if constexpr (KS > 1) {
          o = part[wave][4 * i + q][lane];
#pragma unroll
          for (int k = 1; k < KS; ++k) o += part[k * NS + wave][4 * i + q][lane];
        } else {
          o = f32x4{yv[i][j][4 * q], yv[i][j][4 * q + 1], yv[i][j][4 * q + 2], yv[i][j][4 * q + 3]};
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float ov = o[e] + bv;
          if (epi.R > 0) ov += r[4 * q + e] * epi.lora_scale;
          if constexpr (decltype(ACT)::value == MLXQ_ACT_GELU_EXACT) ov = gelu_erf(ov);
          else if constexpr (decltype(ACT)::value == MLXQ_ACT_GELU_TANH) ov = gelu_tanh<false>(ov);
          const int row = 32 * i + 8 * q + 4 * half + e;
          const uint32_t at = n_ok ? (uint32_t)(row * N + n) * 4u : 0xfffffffcu;  // rows past M fall past the resource
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(ov), ry, at, 0, 0);
        }
      }
    }
  };
  if (epi.act == MLXQ_ACT_GELU || epi.act == MLXQ_ACT_GELU_EXACT) finish(std::integral_constant<int, MLXQ_ACT_GELU_EXACT>{});
  else if (epi.act == MLXQ_ACT_GELU_TANH) finish(std::integral_constant<int, MLXQ_ACT_GELU_TANH>{});
  else finish(std::integral_constant<int, MLXQ_ACT_NONE>{});
}

template <typename XT, typename SB, int BITS, int GS, int BM, int KS, int TN = 1>
static int launch_strip(const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* s, const void* b,
                        int64_t N, void* y, const F32Epilogue& epi, hipStream_t st) {
  constexpr int BN = 256 / KS * TN;
  const int64_t tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  if (tiles > 0x7fffffff) return set_error(MLXQ_EINVAL, "qmm_f32: problem too large");
  hipLaunchKernelGGL((qmm_f32_strip_kernel<XT, SB, BITS, GS, BM, KS, TN>), dim3((unsigned)tiles), dim3(512), 0, st,
                     (const XT*)x, M, K, wq, (const SB*)s, (const SB*)b, N, (float*)y, epi);
  return check_launch("qmm_f32");
}

// Tile height and K-groups: 0: 128 rows; 1: 64 rows; 2: 64 rows in 2 K-groups; 3: 32 rows in 4.
// One workgroup runs per CU (512 threads at 141 registers or more, or 84 KB of LDS or more: a second one fits
// beside none of the four), so a shape costs its rounds of tiles times its chain of K steps: the
// shape with the least rounds * (steps * t + 5 us), with t, the measured time of a step (us), 0.95 /
// 0.63 / 0.71 / 0.63 for one pass and 1.7 / 0.95 / 1.2 / 1.25 for two.  Measured, us for shapes 0..3
// (Q4 g64 unless stated): fp16 77 x 1280 x 5120 Q8 26.4 / 19.1 / 13.9 / 9.3, 77 x 5120 x 1280 81.7 /
// 55.4 / 33.8 / 17.1, 256 x 1280 x 5120 25.9 / 18.3 / 13.9 / 21.9, 512 x 3072 x 3072 52.7 / 36.1 / 25.1 /
// 39.8, 2048 x 1280 x 1280 26.7 / 19.1 / 25.4 / 35.1, 1024 x 1280 x 10240 54.0 / 54.9 / 64.3 / 132;
// f32 20 x 3072 x 12288 82.8 / 47.5 / 33.6 / 19.9, 256 x 3072 x 3072 86.4 / 51.6 / 34.8 / 38.0,
// 512 x 3072 x 12288 90.1 / 108 / 115 / 213, 1024 x 3072 x 3072 88.3 / 53.4 / 71.3 / 107.
inline int strip_shape(int64_t M, int64_t K, int64_t N, int gs, bool two_pass) {
  static constexpr int kRows[4] = {128, 64, 64, 32}, kGroups[4] = {1, 1, 2, 4};
  static constexpr int kStep[2][4] = {{95, 63, 71, 63}, {170, 95, 120, 125}};  // 10 ns
  if (K >= kStripReach / 2 || N >= kStripReach / 2) return 1;  // 32-bit offsets within a tile
  const int64_t cus = device_cu_count(), steps = K / 64;
  int best = 0;
  int64_t best_cost = 0;
  for (int i = 0; i < 4; ++i) {
    const int64_t bn = 256 / kGroups[i];
    if (i > 1 && steps / (gs == 128 ? 2 : 1) < kGroups[i]) continue;  // every K-group needs a step
    const int64_t tiles = ((M + kRows[i] - 1) / kRows[i]) * ((N + bn - 1) / bn);
    const int64_t cost = (tiles + cus - 1) / cus * ((steps + kGroups[i] - 1) / kGroups[i] * kStep[two_pass][i] + 500);
    if (i == 0 || cost < best_cost) {
      best = i;
      best_cost = cost;
    }
  }
  return best;
}

template <typename XT, typename SB, int BITS, int GS>
static int strip_tile(const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* s, const void* b, int64_t N,
                      void* y, const F32Epilogue& epi, hipStream_t st) {
  switch (strip_shape(M, K, N, GS, std::is_same<XT, float>::value)) {
    case 0:
      // f32 activations, Q4, more than a round and a half of tiles: 64 x 512 instead of 128 x 256, two
      // strips per wave: half the LDS reads of activations, for twice the code conversions, which two passes'
      // MFMAs hide.  Same-process A/B, 128 x 256 ->
      // 64 x 512: 4608 x 3072 x 12288 694 -> 648 us, 4608 x 12288 x 3072 748 -> 713, 4608 x 3072 x 3072
      // g128 175 -> 164; 1024 x 3072 x 12288 (1.5 rounds) 171 -> 174.  Q8 needs twice the weight
      // registers and spills (4608 x 3072 x 9216 597 -> 630).  fp16 has one pass and loses by the
      // conversions (4096 x 1280 x 10240 152 -> 166, 2048 x 3072 x 12288 190 -> 204; 233 registers, no spill).
      if constexpr (std::is_same<XT, float>::value && BITS == 4) {
        if (((M + 63) / 64) * ((N + 511) / 512) * 2 > device_cu_count() * 3)
          return launch_strip<XT, SB, BITS, GS, 64, 1, 2>(x, M, K, wq, s, b, N, y, epi, st);
      }
      return launch_strip<XT, SB, BITS, GS, 128, 1>(x, M, K, wq, s, b, N, y, epi, st);
    case 1: return launch_strip<XT, SB, BITS, GS, 64, 1>(x, M, K, wq, s, b, N, y, epi, st);
    case 2: return launch_strip<XT, SB, BITS, GS, 64, 2>(x, M, K, wq, s, b, N, y, epi, st);
    default: return launch_strip<XT, SB, BITS, GS, 32, 4>(x, M, K, wq, s, b, N, y, epi, st);
  }
}

template <typename XT, typename SB>
static int strip_bits_gs(const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* s, const void* b,
                         int64_t N, int gs, int bits, void* y, const F32Epilogue& epi, hipStream_t st) {
#define MLXQ_ST(B, G)                                          \
  if constexpr (!(std::is_same<XT, float>::value && G == 32)) \
    if (bits == B && gs == G) return strip_tile<XT, SB, B, G>(x, M, K, wq, s, b, N, y, epi, st);
  MLXQ_ST(4, 32) MLXQ_ST(4, 64) MLXQ_ST(4, 128) MLXQ_ST(8, 32) MLXQ_ST(8, 64) MLXQ_ST(8, 128)
#undef MLXQ_ST
  return set_error(MLXQ_EINVAL, "qmm_f32: unsupported bits=%d group_size=%d", bits, gs);
}

// One operand mix per translation unit (qmm_f32_strip_*.hip), so that they compile side by side.
#define MLXQ_STRIP_ENTRY(NAME, XT, SB)                                                                          \
  int NAME(const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* s, const void* b, int64_t N,    \
           int gs, int bits, void* y, const F32Epilogue& epi, hipStream_t st) {                                 \
    return strip_bits_gs<XT, SB>(x, M, K, wq, s, b, N, gs, bits, y, epi, st);                                   \
  }
int run_strip_f32_bf16(const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* s, const void* b, int64_t N,
                       int gs, int bits, void* y, const F32Epilogue& epi, hipStream_t st);
int run_strip_f32_f32(const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* s, const void* b, int64_t N,
                      int gs, int bits, void* y, const F32Epilogue& epi, hipStream_t st);
int run_strip_f16_bf16(const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* s, const void* b, int64_t N,
                       int gs, int bits, void* y, const F32Epilogue& epi, hipStream_t st);
int run_strip_f16_f32(const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* s, const void* b, int64_t N,
                      int gs, int bits, void* y, const F32Epilogue& epi, hipStream_t st);
int run_strip_bf16_f32(const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* s, const void* b, int64_t N,
                       int gs, int bits, void* y, const F32Epilogue& epi, hipStream_t st);

}  // namespace mlxq
