// qmv_mfma.h — decode GEMV y[M,N] = x[M,K] . W^T for M <= 8 on gfx950 matrix cores.
//
// Two kernels: the 16-row tile kernel described here (M = 2..8, Q8, and K not a multiple of
// 1024), and, further down, the one-row kernel that serves M = 1 with Q4 codes (one weight row per
// wave, no split-K reduction).  Both compute the same exact-f32 factored form.
//
// The path is HBM-bound and small (a few MB per call), so the kernel is built around the load
// shape the memory system streams best and around latency: every 16-byte weight load a wave
// needs is issued up front, each load covers 16 rows x 64 contiguous bytes (4 lanes per row), the
// packed codes go straight into MFMA operand registers, and each load step is folded as soon as
// its data arrives (the step code is branch-free, so the compiler waits for one load per step).
//
// Semantics are the exact-f32 factored form (no bf16 rounding of dequantized weights):
//   y[m,n] = sum_g ( s[n,g] * sum_{k in g} x[m,k]*c[n,k]  +  b[n,g] * X[m,g] ),  X = sum_{k in g} x.
// Q4 codes enter the MFMA as exact bf16 values c, two per fp8 scaled convert (unpack_q4), and
// Q8 codes as bf16(c) (exact for c < 256); both fold per group as y += s*acc + b*X.
// X comes from the same activation fragments multiplied by an all-ones operand on the MFMA.
//
// v_mfma_f32_16x16x32_bf16 with A = activations (rows m = lane&15; rows >= M read row 0 and are
// never stored) and B = weights (columns n = lane&15).  Lane quarter q = lane>>4 holds the 16
// bytes [16q, 16q+16) of the row's 64-byte load step: 32 Q4 codes (4 words) or 16 Q8 codes.
// Each MFMA takes one 8-code run per lane, and all four runs of one MFMA must lie in one group:
//   * Q8 (64 codes per step): MFMA j takes words 2j, 2j+1 of every lane — one 64-code block.
//   * Q4, group 128 (128 codes per step, one group): MFMA i takes word i of every lane.
//   * Q4, group 64: lanes q = 0,1 hold group 2t and lanes q = 2,3 group 2t+1.  Two
//     v_permlane32_swap ops exchange words 2,3 of the low lane half with words 0,1 of the high
//     half, after which words 0,1 of every lane belong to group 2t and words 2,3 to group 2t+1.
//   * Q8, group 32: lanes q = 0,1 hold group 2t and q = 2,3 group 2t+1; the same two swaps as
//     for Q4 group 64 make words 0,1 (MFMA 0) group 2t and words 2,3 (MFMA 1) group 2t+1.
//   * Q4, group 32: lane quarter q holds group 4t+q whole.  The same two swaps followed by two
//     v_permlane16_swap ops (odd 16-lane rows against even rows) transpose the 4 x 4 block of
//     (quarter, word), after which word i of every lane belongs to group 4t+i.
// Each lane reads the activation run matching its code run from LDS (per-lane offsets below).
// The 16x16 result holds column n = lane&15 for rows m = 4q + e.
// A workgroup owns up to 16 weight rows (one MFMA tile); its waves split K and reduce through LDS
// at the end.
// Q4 k-order inside an 8-run is [0,2,4,6,1,3,5,7] (low nibbles first, see unpack_q4); the
// activation rows are permuted to match with v_perm_b32 as they are copied into LDS.
#pragma once

#include <atomic>
#include <type_traits>
#include <utility>

#include "mlxq_common.h"

namespace mlxq {

namespace {

constexpr int kBufferFlags = 0x00020000;
constexpr int kMaxWaves = 16;  // waves per workgroup (they split K)
constexpr int kCopySlots = 8;  // 16-byte activation chunks a lane stages (registers), all rows
constexpr int kMaxLds = 160 * 1024;
constexpr uint32_t kOob = 0x7ffffff0u;  // buffer offset past every resource: loads return zero

// Q4 word (codes c0..c7, c_i at bits 4i) -> bf16 pairs (c0, c2), (c4, c6), (c1, c3), (c5, c7).
// The low and high nibbles are split into bytes once; a byte c <= 15 read as OCP fp8 E4M3 is
// exactly c * 2^-9, so v_cvt_scalef32_pk_bf16_fp8 with scale 2^9 turns two code bytes into two
// exact bf16 values.
__device__ __forceinline__ bf16x8 unpack_q4(uint32_t w) {
  const uint32_t lo = w & 0x0f0f0f0fu;          // bytes c0, c2, c4, c6
  const uint32_t hi = (w >> 4) & 0x0f0f0f0fu;   // bytes c1, c3, c5, c7
  u32x4 o;
  o[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, false));
  o[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, true));
  o[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, false));
  o[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, true));
  return __builtin_bit_cast(bf16x8, o);
}

// Activation run x0..x7 (raw bf16 pairs r0..r3) -> order [0,2,4,6,1,3,5,7], matching unpack_q4.
__device__ __forceinline__ u32x4 perm_q4(u32x4 r) {
  u32x4 o;
  o[0] = __builtin_amdgcn_perm(r[1], r[0], 0x05040100u);
  o[1] = __builtin_amdgcn_perm(r[3], r[2], 0x05040100u);
  o[2] = __builtin_amdgcn_perm(r[1], r[0], 0x07060302u);
  o[3] = __builtin_amdgcn_perm(r[3], r[2], 0x07060302u);
  return o;
}

// Two Q8 words (codes c0..c7 in natural order) -> bf16(c).
__device__ __forceinline__ bf16x8 cvt_q8(uint32_t w0, uint32_t w1) {
  u32x4 o;
  o[0] = pack_bf16x2((float)(w0 & 0xffu), (float)((w0 >> 8) & 0xffu));
  o[1] = pack_bf16x2((float)((w0 >> 16) & 0xffu), (float)(w0 >> 24));
  o[2] = pack_bf16x2((float)(w1 & 0xffu), (float)((w1 >> 8) & 0xffu));
  o[3] = pack_bf16x2((float)((w1 >> 16) & 0xffu), (float)(w1 >> 24));
  return __builtin_bit_cast(bf16x8, o);
}

__device__ __forceinline__ u32x4 load16(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// Raw buffer resource over `bytes` bytes at p: loads at offsets past the end return zero.
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const T* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(p), (short)0, bytes, kBufferFlags);
}

// v_permlane32_swap_b32: lanes 32..63 of `lo_keep` trade places with lanes 0..31 of `hi_keep`.
// Afterwards lanes 0..31 still hold their own `lo_keep` and lanes 32..63 their own `hi_keep`.
__device__ __forceinline__ void swap_lane_halves(uint32_t& lo_keep, uint32_t& hi_keep) {
  const auto r = __builtin_amdgcn_permlane32_swap(lo_keep, hi_keep, false, false);
  lo_keep = r[0];
  hi_keep = r[1];
}

// v_permlane16_swap_b32: the odd 16-lane rows (1, 3) of `even_keep` trade places with the even
// rows (0, 2) of `odd_keep`; row 2k keeps its own `even_keep`, row 2k + 1 its own `odd_keep`.
__device__ __forceinline__ void swap_lane_rows(uint32_t& even_keep, uint32_t& odd_keep) {
  const auto r = __builtin_amdgcn_permlane16_swap(even_keep, odd_keep, false, false);
  even_keep = r[0];
  odd_keep = r[1];
}

// Row pitch in floats of the per-row (s, zc) pair table in LDS: at least 2G, a multiple of 4 (the
// fold reads 16 bytes) and an odd multiple of 4, so the 16 rows read in one step (one per lane)
// land on 16 distinct 16-byte bank quads.  A pitch of exactly 2G puts every row on the same banks
// whenever 2G is a multiple of 64 (K = 8192, group 64: a 16-way conflict on every fold).
__host__ __device__ constexpr int sz_pitch(int G) {
  const int p = (2 * G + 3) & ~3;
  return (p & 4) ? p : p + 4;
}

// Whether a tile of `steps` load steps per wave and MR activation rows stays within the 128
// registers per lane of a 1024-thread workgroup (the counts the compiler reports for these
// kernels): 8 steps only with one row, and for Q4 with group 64 (two groups per step) 6 steps
// with at most two rows.  Larger combinations spilled (and spills doubled a launch's time).
constexpr bool qmv_steps_fit(int bits, int gs, int steps, int mr) {
  return !(steps == 8 && mr > 1) && !(bits == 4 && gs == 64 && steps == 6 && mr > 2) &&
         !(gs == 32 && steps > 4);
}

}  // namespace

// Scale/bias group slots one wave keeps: the groups its load steps touch (a group 128 of Q8 spans
// two steps and may straddle two waves, hence the spare slot).
__host__ __device__ constexpr int qmv_wave_groups(int bits, int gs, int steps) {
  return bits == 8 ? (gs == 128 ? (steps + 2) / 2 : steps * (64 / gs)) : steps * (128 / gs);
}

// Bytes of LDS one wave owns: its activation rows (M rows of steps * 64 bytes of codes' worth of
// activations, padded so rows start on different banks) and its (s, zc) table.
__host__ __device__ constexpr int qmv_wave_lds(int bits, int gs, int steps, int M) {
  return M * (steps * (512 / bits) * 2 + 16) + 16 * sz_pitch(qmv_wave_groups(bits, gs, steps)) * 4;
}

// One 16-row GEMV tile as seen by one wave: the wave's K range of T load steps, the operand
// registers between the issue of its loads and their use, and its private LDS region.  The
// weights pass through a ring of STEPS load registers: the first STEPS steps are issued up front
// and each register is reloaded with step d + STEPS as soon as step d's MFMAs have read it (T = 2
// STEPS reaches twice the K of one register round at the same register count).  The last wave's
// range may run past K: its activations there load as zero (so those steps' products and group
// sums are zero, whatever codes the weight loads find past the row's end) and so do the scales
// and biases of groups past the row's end.
// Contract of every kernel built from it (checked on the host by qmv_plan):
// 1 <= M <= MR, K % group == 0, bf16 scales and biases, the row's
// load steps (ceil(K*BITS/512)) covered by the waves of one matrix (T each, the last wave's range may end
// past K), dynamic LDS of at least the operands and the partial sums (QmvPlan::lds, qmv_multi_lds), every
// buffer < 2 GiB.
template <int BITS, int GS, int STEPS, int MR, int T>
struct GemvTile {
  static_assert(T >= STEPS, "ring shorter than the wave's steps");
  static constexpr int CPL = 512 / BITS;          // codes per row in one 64-byte load step
  static constexpr bool G64 = GS == 64, G32 = GS == 32;
  static constexpr bool Q4G32 = BITS == 4 && G32;  // four groups per step, one per lane quarter
  // two groups per step, one per lane half (Q4 group 64, Q8 group 32)
  static constexpr bool PAIR = (BITS == 4 && G64) || (BITS == 8 && G32);
  static constexpr int NACC = Q4G32 ? 4 : 2;      // group accumulators per load step
  static constexpr int NM = BITS == 4 ? 4 : 2;    // MFMAs per load step
  static constexpr int E = MR < 4 ? MR : 4;       // result registers per lane that can hold a row < M
  static constexpr int XCH = T * CPL / 8;         // 16-byte activation chunks per row in the wave's range
  static constexpr int XSL = (XCH + 63) / 64;     // ... per lane
  static constexpr int XB = kCopySlots / XSL < MR ? (kCopySlots / XSL > 0 ? kCopySlots / XSL : 1) : MR;  // rows staged at a time
  static constexpr int NGW = qmv_wave_groups(BITS, GS, T);
  static constexpr int PW = sz_pitch(NGW);        // (s, zc) table row pitch, floats
  static constexpr int SBL = (16 * NGW + 63) / 64;  // scale entries per lane
  static constexpr int XW = T * CPL * 2 + 16;       // LDS pitch of the wave's activation rows

  int lane, c16, q, M, K, N, G, ls0, kb, g0;
  unsigned char* wl;  // this wave's LDS region: activation rows, then the (s, zc) table
  float* szw;
  u32x4 cx[XB][XSL];
  uint32_t cs[SBL], cz[SBL];
  u32x4 wv[STEPS];
  __amdgpu_buffer_rsrc_t rw;
  uint32_t w_base;

  // wave_all: the wave's index in the workgroup (selects its LDS region); wave: its index among
  // the waves of its matrix (selects its K range).  A tile is the rows [n0, n0 + nr) of an [N, K]
  // matrix, nr <= 16 (MFMA columns past nr load nothing and are never stored).
  __device__ __forceinline__ GemvTile(int lane_, int wave_all, int wave, int M_, int K_, int N_, unsigned char* lds) {
    lane = lane_;
    c16 = lane & 15;
    q = lane >> 4;
    M = M_;
    K = K_;
    N = N_;
    G = K / GS;
    ls0 = wave * T;
    kb = ls0 * CPL;
    g0 = kb / GS;
    wl = lds + wave_all * (M * XW + 16 * PW * 4);
    szw = reinterpret_cast<float*>(wl + M * XW);
  }

  // The wave's activation range as 16-byte chunks (out-of-range chunks read as zero), rows m0 ..
  // m0 + XB - 1.
  __device__ __forceinline__ void issue_x(__amdgpu_buffer_rsrc_t rx, int m0) {
#pragma unroll
    for (int i = 0; i < XB; ++i) {
      if (m0 + i < M) {
#pragma unroll
        for (int j = 0; j < XSL; ++j) {
          const int c = lane + 64 * j;
          cx[i][j] = load16(rx, c < XCH && kb + c * 8 < K ? (uint32_t)(((m0 + i) * K + kb + c * 8) * 2) : kOob);
        }
      }
    }
  }

  // The scale and bias of each (row, group) slot the wave folds.
  __device__ __forceinline__ void issue_sb(__amdgpu_buffer_rsrc_t rs, __amdgpu_buffer_rsrc_t rz, int n0, int nr) {
#pragma unroll
    for (int j = 0; j < SBL; ++j) {
      const int e = lane + 64 * j;
      const int r = e / NGW, gl = e - r * NGW;  // constant divisor
      const bool ok = e < 16 * NGW && r < nr && g0 + gl < G;
      const uint32_t off = ok ? ((uint32_t)(n0 + r) * (uint32_t)G + (uint32_t)(g0 + gl)) * 2u : kOob;
      cs[j] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(rs, off, 0, 0);
      cz[j] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(rz, off, 0, 0);
    }
  }

  // Weight loads: 16 rows x 64 contiguous bytes per load; the lanes of rows past the tile's nr read
  // past every buffer (zero, no memory traffic).
  __device__ __forceinline__ uint32_t w_offset(int n0, int nr) const {
    return c16 < nr ? (uint32_t)(n0 + c16) * (uint32_t)(K * BITS / 8) + (uint32_t)(ls0 * 64 + q * 16) : kOob;
  }
  // The first tile's first STEPS.
  __device__ __forceinline__ void issue_w(__amdgpu_buffer_rsrc_t rw_, int n0, int nr) {
    rw = rw_;
    w_base = w_offset(n0, nr);
#pragma unroll
    for (int d = 0; d < STEPS; ++d) wv[d] = load16(rw, w_base + (uint32_t)d * 64u);
  }

  // Operands into the wave's LDS region.  Q4 activation runs are stored permuted to
  // [0,2,4,6,1,3,5,7] so they pair with the unpacked code layout; scales and biases become
  // f32 pairs (s, b), ready for the fold.  Only this wave reads them back, so a wave-level ordering
  // point (publish) replaces a workgroup barrier.
  __device__ __forceinline__ void stage_x(int m0) {
#pragma unroll
    for (int i = 0; i < XB; ++i) {
      if (m0 + i < M) {
#pragma unroll
        for (int j = 0; j < XSL; ++j) {
          const int c = lane + 64 * j;
          if (c < XCH)
            *reinterpret_cast<u32x4*>(wl + (m0 + i) * XW + c * 16) = BITS == 4 ? perm_q4(cx[i][j]) : cx[i][j];
        }
      }
    }
  }
  __device__ __forceinline__ void stage_sb() {
#pragma unroll
    for (int j = 0; j < SBL; ++j) {
      const int e = lane + 64 * j;
      if (e < 16 * NGW) {
        const int r = e / NGW, gl = e - r * NGW;
        const float sv = __uint_as_float(cs[j] << 16), zv = __uint_as_float(cz[j] << 16);
        *reinterpret_cast<f32x2*>(szw + r * PW + 2 * gl) = f32x2{sv, zv};
      }
    }
  }
  __device__ __forceinline__ void publish() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
  }

  // Per load step: NM MFMAs x . codes and NM MFMAs x . ones (group sums), then the fold of
  // each group, y += s*acc + zc*X.  yacc[e] is result row 4q + e of column c16.  NEXT: the workgroup
  // walks several tiles, and the next one's weights start at w_next (kOob past the last: loads there
  // return zero without memory traffic).
  template <bool NEXT>
  __device__ __forceinline__ void fold(float (&yacc)[E], uint32_t w_next) {
    const unsigned char* xa[NM];  // this lane's activation run for MFMA i at the wave's first step
#pragma unroll
    for (int i = 0; i < NM; ++i) {
      int k;
      if constexpr (BITS == 8 && G32) k = (q < 2 ? 16 * q : 16 * (q - 2) + 8) + 32 * i;
      else if constexpr (BITS == 8) k = 16 * q + 8 * i;
      else if constexpr (G32) k = 32 * i + 8 * q;  // after the word transpose: MFMA i = group i
      else if constexpr (!G64) k = 32 * q + 8 * i;
      else if (i < 2) k = (q < 2 ? 32 * q : 32 * (q - 2) + 16) + 8 * i;
      else k = (q < 2 ? 64 + 32 * q : 32 * q + 16) + 8 * (i - 2);
      xa[i] = wl + (c16 < M ? c16 : 0) * XW + k * 2;
    }
    const float* sz = szw + c16 * PW;
    bf16x8 ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = (__bf16)1.0f;
#pragma unroll
    for (int e = 0; e < E; ++e) yacc[e] = 0.0f;

    auto fold1 = [&](const f32x4& acc, const f32x4& xsum, float s, float zc) {
#pragma unroll
      for (int e = 0; e < E; ++e) yacc[e] = fmaf(s, acc[e], fmaf(zc, xsum[e], yacc[e]));
    };

    // Activation runs: every lane reads, lanes of A rows c16 >= M the run of row 0 (an A row
    // m >= M only feeds result row m, which is never stored).  The 16 lanes of a quarter then read
    // at most M distinct addresses (broadcast); a read restricted to the lanes of rows < M cost
    // the compiler ten 64-bit register copies per step to keep the other lanes' operands.
    using SZ = typename std::conditional<PAIR, f32x4, f32x2>::type;
    bf16x8 a[T][NM];
    SZ p[T];
    f32x4 p32[T][2];  // group 32: the (s, zc) pairs of the step's four groups
    f32x4 acc[T][NACC], xsum[T][NACC];

    // A step's LDS operands: its activation runs and its (s, zc) pairs.
    auto read_step = [&](int d) {
#pragma unroll
      for (int i = 0; i < NM; ++i) a[d][i] = *reinterpret_cast<const bf16x8*>(xa[i] + d * (CPL * 2));
      if constexpr (Q4G32) {
        p32[d][0] = *reinterpret_cast<const f32x4*>(sz + 8 * d);  // groups 4ls, 4ls+1
        p32[d][1] = *reinterpret_cast<const f32x4*>(sz + 8 * d + 4);  // groups 4ls+2, 4ls+3
      } else if constexpr (PAIR) {
        p[d] = *reinterpret_cast<const f32x4*>(sz + 4 * d);  // groups 2ls, 2ls+1
      } else {
        // Q4/128 and Q8/64: one group per step; Q8/128: a group every two steps
        const int gl = (BITS == 4 || G64) ? d : ((ls0 + d) >> 1) - g0;
        p[d] = *reinterpret_cast<const f32x2*>(sz + 2 * gl);
      }
    };
    // A step's products: NM MFMAs x . codes and NM MFMAs x . ones (the group sums); then the ring
    // register is reloaded with step d + STEPS.
    auto mfma_step = [&](int d) {
      const int slot = d % STEPS;
      uint32_t w[4] = {wv[slot][0], wv[slot][1], wv[slot][2], wv[slot][3]};
      if constexpr (PAIR) {  // Q8 group 32: words 0,1 and 2,3 are its two MFMAs' pairs
        swap_lane_halves(w[0], w[2]);
        swap_lane_halves(w[1], w[3]);
      } else if constexpr (Q4G32) {
        // Quarter q's 16 bytes are group q of the step (words = 8-code runs).  Transpose the
        // 4 x 4 (quarter, word) block: afterwards word i of quarter q is run q of group i, so
        // MFMA i covers group i alone.
        swap_lane_halves(w[0], w[2]);
        swap_lane_halves(w[1], w[3]);
        swap_lane_rows(w[0], w[1]);
        swap_lane_rows(w[2], w[3]);
      }
#pragma unroll
      for (int h = 0; h < NACC; ++h) {
        acc[d][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        xsum[d][h] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      }
#pragma unroll
      for (int i = 0; i < NM; ++i) {
        const int h = (Q4G32 || (BITS == 8 && G32)) ? i : ((BITS == 4 && G64) ? i >> 1 : 0);
        const bf16x8 b = BITS == 4 ? unpack_q4(w[i]) : cvt_q8(w[2 * i], w[2 * i + 1]);
        acc[d][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[d][i], b, acc[d][h], 0, 0, 0);
        xsum[d][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[d][i], ones, xsum[d][h], 0, 0, 0);
      }
      // The register's next load: this tile's step d + STEPS, or the next tile's d + STEPS - T.
      if (d + STEPS < T) {
        wv[slot] = load16(rw, w_base + (uint32_t)(d + STEPS) * 64u);
      } else if constexpr (NEXT) {
        __builtin_amdgcn_sched_barrier(0);
        wv[slot] = load16(rw, w_next + (uint32_t)(d + STEPS - T) * 64u);
      }
    };
    // A step's fold into the result.  The result is pinned after each fold: otherwise the
    // compiler sinks every fold below the last step and keeps all steps' products live at once.
    auto fold_step = [&](int d) {
      if constexpr (Q4G32) {
        fold1(acc[d][0], xsum[d][0], p32[d][0][0], p32[d][0][1]);
        fold1(acc[d][1], xsum[d][1], p32[d][0][2], p32[d][0][3]);
        fold1(acc[d][2], xsum[d][2], p32[d][1][0], p32[d][1][1]);
        fold1(acc[d][3], xsum[d][3], p32[d][1][2], p32[d][1][3]);
      } else if constexpr (PAIR) {
        fold1(acc[d][0], xsum[d][0], p[d][0], p[d][1]);
        fold1(acc[d][1], xsum[d][1], p[d][2], p[d][3]);
      } else {
        fold1(acc[d][0], xsum[d][0], p[d][0], p[d][1]);
      }
#pragma unroll
      for (int e = 0; e < E; ++e) asm volatile("" : "+v"(yacc[e]));
    };

    // Software pipeline over the steps: iteration d reads step d+1's LDS operands, runs step d's
    // MFMAs (waiting for its weight load only) and folds step d-1, whose products have completed
    // meanwhile, so the LDS-read and MFMA latencies of consecutive steps overlap.  Scheduling
    // fences between iterations keep at most two steps' operands live.
    read_step(0);
#pragma unroll
    for (int d = 0; d < T; ++d) {
      __builtin_amdgcn_sched_barrier(0);
      if (d + 1 < T) read_step(d + 1 < T ? d + 1 : d);
      mfma_step(d);
      if (d > 0) fold_step(d - 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    fold_step(T - 1);
    w_base = w_next;
  }
};

// The bf16 epilogue of a linear on its rounded product: the dense bias and a bf16 activation's table
// (each null when absent), one rounding per op.
__device__ __forceinline__ uint16_t gemv_finish(float v, int n, const uint16_t* __restrict__ bias,
                                                const uint16_t* __restrict__ act_table) {
  if (bias) v = round_bf16(v) + bf16_bits_to_f32(bias[n]);
  const uint16_t h = f32_to_bf16_bits(v);
  return act_table ? act_table[h] : h;
}

// The GEMV launch: workgroup b owns `rows` consecutive weight rows, one tile of up to 16 or (MULTI)
// several, 16 at a time; its waves split K.  NMAT = 2 is the SwiGLU decode form: the second wave half
// streams the same rows of a second matrix (up).
// Each wave stages only its own operands (its K range of the activations once, the scales and biases
// of its groups per tile) into its own LDS region, so it starts on its weights as soon as its own
// operands land; the only workgroup barrier per tile is that of the split-K reduction, whose partial
// sums alternate between two buffers.  MULTI: a weight register is reloaded with the next tile's step
// as soon as its MFMAs have read it, so the weight stream runs on through the reductions; with one
// tile per workgroup the stream ramps up and drains for each 16 rows and the activations are fetched
// anew for them (M = 5, K = 4096: 80 KB of activations per 64 KB of weights).  The decode MLP 4096 /
// 11008 at M = 5: 30.3 -> 20.7 us, with the down projection's five rows in one launch instead of two.
template <int BITS, int GS, int STEPS, int MR, int NMAT, int RING, bool MULTI>
__device__ __forceinline__ void qmv_mfma_body(
    const uint16_t* __restrict__ x, int M, int K, const uint32_t* __restrict__ wq,
    const uint16_t* __restrict__ scales, const uint16_t* __restrict__ biases,
    const uint32_t* __restrict__ wq2, const uint16_t* __restrict__ scales2,
    const uint16_t* __restrict__ biases2, int N, int rows, uint16_t* __restrict__ y,
    const uint16_t* __restrict__ bias, const uint16_t* __restrict__ act_table) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int NT = blockDim.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int W = (NT >> 6) / NMAT;  // waves per matrix
  const int mat = NMAT == 1 ? 0 : __builtin_amdgcn_readfirstlane(wave_all / W);
  const int n_begin = blockIdx.x * rows;
  const int n_end = N - n_begin < rows ? N : n_begin + rows;
  using Tile = GemvTile<BITS, GS, STEPS, MR, STEPS * RING>;
  Tile t(lane, wave_all, wave_all - mat * W, M, K, N, lds);
  // Partial sums [wave][row m][17]: over the operands, all 16 rows, or (MULTI) in two buffers past them, the
  // rows below MR.  One tile stores every row, unconditionally: with only the lanes of rows below MR storing,
  // the compiler tracked the fold for those lanes and took up to 11 more registers (64 -> 68 for Q4 group 32,
  // two steps, two rows), one workgroup per CU instead of two: [2, 1792] SwiGLU 6784 5.7 -> 6.4 us.
  constexpr int RR = MULTI ? MR : 16;
  float* const red0 = reinterpret_cast<float*>(lds + (MULTI ? (NT >> 6) * (M * Tile::XW + 16 * Tile::PW * 4) : 0));
  const int red_buf = (NT >> 6) * MR * 17;
  const int sb_total = (int)(((uint32_t)N * (uint32_t)t.G * 2u + 3u) & ~3u);  // whole dwords
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(x, M * K * 2), rs = make_rsrc(mat ? scales2 : scales, sb_total),
                               rz = make_rsrc(mat ? biases2 : biases, sb_total);
  auto rows_at = [&](int n0) { return n_end - n0 < 16 ? n_end - n0 : 16; };
  t.issue_x(rx, 0);
  t.issue_sb(rs, rz, n_begin, rows_at(n_begin));
  // The weight streams are issued once every wave of the workgroup has issued its operand
  // loads: a CU's vector memory requests are served in order, and a wave whose small operand
  // loads queue behind its neighbours' weight streams waits microseconds for them.  (A bare
  // s_barrier: nothing here waits for the loads themselves.)  The SwiGLU launch skips it (8.27 ->
  // 8.02 us without it on the decode shape; the one-matrix launches are unchanged either way).
  if constexpr (NMAT == 1) __builtin_amdgcn_s_barrier();
  t.issue_w(make_rsrc(mat ? wq2 : wq, (int)((uint32_t)N * (uint32_t)(K * BITS / 8))), n_begin, rows_at(n_begin));
  t.stage_x(0);
#pragma unroll
  for (int m0 = Tile::XB; m0 < MR; m0 += Tile::XB) {
    if (m0 < M) {
      t.issue_x(rx, m0);
      t.stage_x(m0);
    }
  }
  int buf = 0, n0 = n_begin;
  do {
    t.stage_sb();
    t.publish();
    float yacc[Tile::E];
    const int nn = n0 + 16;
    if constexpr (MULTI) {
      const int nn_rows = nn < n_end ? rows_at(nn) : 0;
      t.issue_sb(rs, rz, nn, nn_rows);
      t.template fold<true>(yacc, t.w_offset(nn, nn_rows));
    } else {
      t.template fold<false>(yacc, 0);
    }
    // Split-K reduction: row 4 q + e of the tile's column c16 (rows past M are never read).
    float* const red = red0 + buf * red_buf;
    const int c16 = lane & 15, q = lane >> 4;
    if constexpr (!MULTI) __syncthreads();
    if (!MULTI || 4 * q < MR) {
#pragma unroll
      for (int e = 0; e < Tile::E; ++e) red[(wave_all * RR + 4 * q + e) * 17 + c16] = yacc[e];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    const int nr = rows_at(n0);
    for (int idx = tid; idx < 16 * M; idx += NT) {  // a one-wave workgroup has 64 < 16*M threads
      const int m = idx >> 4, nl = idx & 15;
      float v = 0.0f;
      for (int w = 0; w < W; ++w) v += red[(w * RR + m) * 17 + nl];
      if constexpr (NMAT == 2) {
        float u = 0.0f;
        for (int w = 0; w < W; ++w) u += red[((W + w) * RR + m) * 17 + nl];
        // each op rounded to bf16 as the reference's separate ops are (qwen3.rs:178-181)
        if (nl < nr) y[m * N + n0 + nl] = f32_to_bf16_bits(silu_bf16(round_bf16(v)) * round_bf16(u));
      } else {
        if (nl < nr) y[m * N + n0 + nl] = gemv_finish(v, n0 + nl, bias, act_table);
      }
    }
    n0 = nn;
    buf ^= 1;
  } while (MULTI && n0 < n_end);
}

// Arguments come first in the order they are needed: 14 dwords of them are preloaded into registers, and
// each further one that a workgroup's first loads wait for costs it a scalar load from memory.  With one
// signature for both forms and the epilogue's operands besides, short launches took 0.1 us longer (2-3 %),
// [2, 1664] x Q8 g128 [31437, 1664]^T 12.4 -> 13.3.
template <int BITS, int GS, int STEPS, int MR, int RING, bool MULTI>
__global__ __launch_bounds__(kMaxWaves * 64) void qmv_mfma_kernel(
    const uint16_t* __restrict__ x, int M, int K, const uint32_t* __restrict__ wq, const uint16_t* __restrict__ scales,
    const uint16_t* __restrict__ biases, int N, int rows, uint16_t* __restrict__ y,
    const uint16_t* __restrict__ bias, const uint16_t* __restrict__ act_table, QmmBatch bat) {
  // Stacked launch: the workgroup's y index selects the matrix (expert).
  if (const int64_t e = blockIdx.y; e > 0) {
    x += e * bat.x;
    wq += e * bat.w;
    scales += e * bat.sb;
    biases += e * bat.sb;
    y += e * bat.y;
    if (bias) bias += e * bat.bias;
  }
  qmv_mfma_body<BITS, GS, STEPS, MR, 1, RING, MULTI>(x, M, K, wq, scales, biases, nullptr, nullptr, nullptr, N, rows, y,
                                                     bias, act_table);
}

template <int BITS, int GS, int STEPS, int MR, int RING, bool MULTI>
__global__ __launch_bounds__(kMaxWaves * 64) void swiglu_mfma_kernel(
    const uint16_t* __restrict__ x, int M, int K, const uint32_t* __restrict__ wq, const uint16_t* __restrict__ scales,
    const uint16_t* __restrict__ biases, const uint32_t* __restrict__ wq2, const uint16_t* __restrict__ scales2,
    const uint16_t* __restrict__ biases2, int N, int rows, uint16_t* __restrict__ y) {
  qmv_mfma_body<BITS, GS, STEPS, MR, 2, RING, MULTI>(x, M, K, wq, scales, biases, wq2, scales2, biases2, N, rows, y,
                                                     nullptr, nullptr);
}

struct QmvPlan {
  int waves, steps, ring, mr, lds, operands;  // waves: all waves of the workgroup (per matrix x matrices)
  int rows;                         // activation rows per launch: M, or 4 or 2 when M is split
};

constexpr int kStepChoices[] = {1, 2, 3, 4, 6, 8};

// Whether a kernel with a ring of `ring` rounds exists: two rounds only with 4..8 load registers
// (and at most two activation rows with group 32, whose four-row ring spilled; more rows split into
// launches of four or two).
constexpr bool qmv_ring_built(int bits, int gs, int steps, int mr, int ring) {
  return ring == 1 || (ring == 2 && (bits == 4 || bits == 8) && steps >= 4 && mr <= (gs == 32 ? 2 : 8));
}

// Whether the several-tiles form exists: where the next tile's operands fit the 128 registers too.
constexpr bool qmv_multi_built(int bits, int gs, int steps, int mr, int nmat, int ring) {
  if (bits == 4 && gs == 32) return ring == 1 && (steps == 1 || (steps == 2 && (nmat == 1 || mr <= 2)));
  if (bits == 4 && gs == 64) return ring == 1 ? steps <= 4 || nmat == 1 : steps == 4 && nmat == 1;
  if (bits == 4 && gs == 128) return !(steps == 8 && ring == 2 && nmat == 2);
  return true;
}

// Picks the load steps per wave: among the counts that divide the row's load steps, fit a
// workgroup of at most kMaxWaves waves, its LDS and its registers (qmv_steps_fit), the one whose
// workgroup comes closest to 12 waves (fewer steps on a tie).  Measured on the decode shapes
// (M = 1..8, K = 3072 and 8192, per-wave operand staging, pipelined fold), 8-12 waves of 3-8 steps
// finish first: a wave starts folding as soon as its own operands arrive, and more, shorter waves
// spread the fold's VALU work (which bounds the last waves' tail) over the SIMDs, while a 16-wave
// workgroup fills a CU on its own (128 registers per wave).  12 against 8: the down GEMV
// (K = 8192) 6.10 -> 5.84 us, gate (K = 3072) 5.40 -> 5.28 us, SwiGLU unchanged; 16 was no better.
//
// A row whose bytes are no multiple of 64 (K = 2880 in Q4: 22.5 load steps) ends inside its last load
// step; the codes past its end are the next row's and fold to zero like those of a padded step.
// Such rows had run on the VALU kernel: [4, 2880] x Q4 g64 [2880, 2880]^T 11.2 -> 4.2 us, [6, 736] x Q8
// g32 [711, 736]^T 11.2 -> 3.7.
//
// When no count divides the row's load steps within those limits (K = 11008: 86 steps of Q4),
// the waves take ceil(steps / waves) each and the last one's range ends past K (cost as above,
// then the fewest padded steps); failing that, each wave takes two rounds of its load registers
// (ring 2: twice the K at the same registers).  one_batch: only plans whose lanes stage all their
// activation chunks at once; a second batch waits for memory again before the wave's first product
// (16 waves of 4 steps in one batch against 11 of 6 in two: [8, 7808] x Q4 g128 [880, 7808]^T 5.4 against
// 6.4 us, SwiGLU [7, 3968] x [7936, 3968]^T 9.7 against 12.5), so the others are for what fits no such plan.  A launch holds its activation rows whole in LDS
// (M x K x 2 bytes), so rows that fit no plan go out as launches of four, else two rows (M = 8,
// K = 18944: four launches of two rows 46 us against 85 us on the VALU GEMV; single rows would
// stream the weights M times and lose to it).
inline bool qmv_plan_rows(int64_t M, int64_t K, int gs, int bits, int nmat, bool one_batch, QmvPlan& p) {
  const int64_t cpl = 512 / bits;
  const int64_t LS = (K + cpl - 1) / cpl;
  const int mr = M <= 1 ? 1 : (M <= 2 ? 2 : (M <= 4 ? 4 : 8));
  for (int pass = 0; pass < 3; ++pass) {  // exact; ragged; ragged with two rounds
    const int ring = pass == 2 ? 2 : 1;
    bool found = false;
    int64_t best_cost = 0, best_pad = 0;
    for (int steps : kStepChoices) {
      if (!qmv_steps_fit(bits, gs, steps, mr) || !qmv_ring_built(bits, gs, steps, mr, ring)) continue;
      const int64_t t = (int64_t)steps * ring;  // load steps per wave
      if (pass == 0 && LS % t != 0) continue;
      const int64_t wpm = (LS + t - 1) / t;
      const int64_t waves = nmat * wpm;
      if (waves > kMaxWaves) continue;
      const int64_t operands = waves * (int64_t)qmv_wave_lds(bits, gs, (int)t, (int)M);
      const int64_t red = waves * 16 * 17 * 4;  // one tile's partial sums
      const int64_t lds = operands > red ? operands : red;
      if (lds > kMaxLds) continue;
      if (one_batch && mr * ((t * cpl / 8 + 63) / 64) > kCopySlots) continue;
      const int64_t cost = waves > 12 ? waves - 12 : 12 - waves;
      const int64_t pad = wpm * t - LS;
      if (found && (cost > best_cost || (cost == best_cost && pad >= best_pad))) continue;
      found = true;
      best_cost = cost;
      best_pad = pad;
      p = {(int)waves, steps, ring, mr, (int)lds, (int)operands, (int)M};
    }
    if (found) return true;
  }
  return false;
}

inline bool qmv_plan(int64_t M, int64_t K, int gs, int bits, int nmat, QmvPlan& p) {
  if (M < 1 || M > 8 || (bits != 4 && bits != 8)) return false;
  if (gs != 32 && gs != 64 && gs != 128) return false;
  if (K <= 0 || K % gs != 0) return false;
  for (bool one_batch : {true, false})
    if (qmv_plan_rows(M, K, gs, bits, nmat, one_batch, p)) return true;
  for (int rows : {4, 2})  // launches of fewer rows
    if (M > rows && qmv_plan_rows(rows, K, gs, bits, nmat, false, p)) return true;
  return false;
}

// Device operands of one launch (the second matrix is used by the SwiGLU form only).
struct QmvArgs {
  const void* x;
  int64_t M, K, N;
  const uint32_t* wq;
  const void *s, *b;
  const uint32_t* wq2;
  const void *s2, *b2;
  void* y;
  const uint16_t* bias = nullptr;       // one matrix: the bf16 epilogue (gemv_finish)
  const uint16_t* act_table = nullptr;
  QmmBatch bat;                         // one matrix: several of the same shape (grid.y)
};

// Rows per workgroup of one tile: 16 for SwiGLU; for one matrix, of 16, 12 and 8 the count whose
// busiest CU streams the fewest rows (the MFMA columns past the count load nothing).  The down
// projection of a decode MLP (N = 3072) takes 12 rows: 256 workgroups, every CU, where 16-row tiles
// left 64 CUs idle.  Stacked experts choose as one of them alone would.
inline int qmv_tile_rows(int64_t N, int nmat) {
  if (nmat == 2) return 16;
  const int64_t cus = device_cu_count();
  int best = 16;
  int64_t best_rows = 0;
  for (int w : {16, 12, 8}) {
    const int64_t rows = ((N + w - 1) / w + cus - 1) / cus * w;
    if (best_rows == 0 || rows < best_rows) {
      best = w;
      best_rows = rows;
    }
  }
  return best;
}

// LDS of a several-tiles workgroup: the operands and two buffers of partial sums.
inline int qmv_multi_lds(const QmvPlan& p) { return p.operands + 2 * p.waves * p.mr * 17 * 4; }

// Rows per workgroup of several tiles, or 0 where one tile each is the better form: the rows spread
// evenly over as many workgroups as the chip holds at once (their waves keep up to 128 registers each,
// 16 waves to a CU).  It takes two whole tiles each to pay, and either activations worth staging once
// (three rows or more) or workgroups of more than 12 waves, which otherwise have a CU to themselves
// and nothing to overlap their start and end.  Same-process A/B, one tile -> several: SwiGLU M = 5,
// 4096 x 11008 17.7 -> 14.6 us, M = 8, 3072 x 8192 11.9 -> 10.1, M = 4 10.1 -> 9.4, but M = 2 8.3 -> 9.0;
// M = 8, 2560 x 9728 g128 11.0 -> 6.4; M = 1 Q8, 4096 x 14336 (16 waves) 17.7 -> 15.4, 3072 x 18432 (12
// waves) 15.4 -> 15.6; 18-22 rows per workgroup 5-6 % slower (M = 4, 2048 x 5120 5.1 -> 5.4).
// Few load steps per wave and tile need more rows: with little of the stream to run on through the
// reductions, 33 to 47 rows are three rounds of tiles as one tile each makes, and the one-tile kernels of so
// few steps are small enough (64 registers) for twice the waves on a CU.  One tile -> several at M < 3 and
// one step: SwiGLU [1, 1024] x Q4 g32 (44 rows) 5.2 -> 6.0 us, (52 rows) 6.0 -> 7.1, [2, 1664] x [8196, 1664]^T (33)
// 5.1 -> 5.5, but [2, 960] x Q8 [28817, 960]^T (113) 12.1 -> 9.8; two: SwiGLU [1, .] Q8 g32 (35) 5.9 -> 6.9,
// [2, 1024] Q8 (48) 6.9 -> 7.5; six and 16 waves: SwiGLU [2, 3072] x Q8 g128 [8064, 3072]^T (32) 9.8 -> 11.3, (50)
// 15.9 -> 15.4, but six and 13 waves, whose one-tile form leaves the CU's other slots empty: [2, 9728] x g128
// [10101, 9728]^T (40) 22.1 -> 13.4, or whose tiles are of 8 rows: [2, 3872] x Q8 g32 [9269, 3872]^T (37) 13.2 ->
// 9.7; eight: (33) 19.4 -> 17.0.  From three rows on, one step: SwiGLU M = 3
// (36) 5.9 -> 6.6, M = 5 (34) 6.5 -> 6.8, M = 8 (34) 7.8 -> 7.4; three or more workgroups to a CU (up to 5
// waves) M = 3 (38) 4.5 -> 4.9, M = 4 (41) 5.3 -> 5.6, M = 8 (40) 7.9 -> 6.5; else M = 3 (37) 5.6 -> 4.6.
inline int qmv_multi_rows(const QmvArgs& a, const QmvPlan& p) {
  if (a.M < 3 && p.waves <= 12) return 0;
  const int lds = qmv_multi_lds(p);
  if (lds > kMaxLds) return 0;
  int64_t per_cu = kMaxWaves / p.waves;
  if (kMaxLds / lds < per_cu) per_cu = kMaxLds / lds;
  const int64_t wgs = device_cu_count() * (per_cu > 0 ? per_cu : 1);
  const int64_t rows = (a.N * a.bat.count + wgs - 1) / wgs;
  const int steps = p.steps * p.ring;
  int64_t least = 32;
  if (a.M < 3) {
    if (steps <= 2) least = a.wq2 != nullptr ? 64 : steps == 1 ? 48 : 40;
    else if (steps < 8 && p.waves == 16 && (a.wq2 != nullptr || qmv_tile_rows(a.N, 1) > 8)) least = 48;
  }
  else if (steps == 1 && a.M < 6 && (a.wq2 != nullptr || per_cu >= 3)) least = 48;
  return rows >= least ? (int)(rows < a.N ? rows : a.N) : 0;
}

template <int BITS, int GS, int STEPS, int MR, int NMAT, int RING, bool MULTI>
static int launch_qmv_mfma(const QmvArgs& a, const QmvPlan& p, int rows, hipStream_t st) {
  // The dynamic-LDS limit is raised once per device (any thread may get here first; setting it
  // twice is harmless).
  static std::atomic<bool> attr_set[64];
  const void* kernel;
  if constexpr (NMAT == 1) kernel = reinterpret_cast<const void*>(&qmv_mfma_kernel<BITS, GS, STEPS, MR, RING, MULTI>);
  else kernel = reinterpret_cast<const void*>(&swiglu_mfma_kernel<BITS, GS, STEPS, MR, RING, MULTI>);
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return set_error(MLXQ_EDEVICE, "qmv: no current device");
  if (dev < 0 || dev >= 64 || !attr_set[dev].load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds) != hipSuccess)
      return set_error(MLXQ_EDEVICE, "qmv: hipFuncSetAttribute failed");
    if (dev >= 0 && dev < 64) attr_set[dev].store(true, std::memory_order_release);
  }
  const dim3 grid((unsigned)((a.N + rows - 1) / rows), (unsigned)a.bat.count), block(p.waves * 64);
  const unsigned lds = MULTI ? qmv_multi_lds(p) : p.lds;
  if constexpr (NMAT == 1)
    hipLaunchKernelGGL((qmv_mfma_kernel<BITS, GS, STEPS, MR, RING, MULTI>), grid, block, lds, st, (const uint16_t*)a.x,
                       (int)a.M, (int)a.K, a.wq, (const uint16_t*)a.s, (const uint16_t*)a.b, (int)a.N, rows,
                       (uint16_t*)a.y, a.bias, a.act_table, a.bat);
  else
    hipLaunchKernelGGL((swiglu_mfma_kernel<BITS, GS, STEPS, MR, RING, MULTI>), grid, block, lds, st, (const uint16_t*)a.x,
                       (int)a.M, (int)a.K, a.wq, (const uint16_t*)a.s, (const uint16_t*)a.b, a.wq2, (const uint16_t*)a.s2,
                       (const uint16_t*)a.b2, (int)a.N, rows, (uint16_t*)a.y);
  return check_launch(NMAT == 2 ? "swiglu_qmv" : "qmv_mfma");
}

template <int BITS, int GS, int STEPS, int MR, int NMAT, int RING>
static int qmv_tiles(const QmvArgs& a, const QmvPlan& p, hipStream_t st) {
  if constexpr (qmv_multi_built(BITS, GS, STEPS, MR, NMAT, RING)) {
    if (const int rows = qmv_multi_rows(a, p))
      return launch_qmv_mfma<BITS, GS, STEPS, MR, NMAT, RING, true>(a, p, rows, st);
  }
  return launch_qmv_mfma<BITS, GS, STEPS, MR, NMAT, RING, false>(a, p, qmv_tile_rows(a.N, NMAT), st);
}

template <int BITS, int GS, int STEPS, int MR, int NMAT>
static int qmv_mr(const QmvArgs& a, const QmvPlan& p, hipStream_t st) {
  if constexpr (qmv_steps_fit(BITS, GS, STEPS, MR)) {
    if (p.ring == 1) return qmv_tiles<BITS, GS, STEPS, MR, NMAT, 1>(a, p, st);
    if constexpr (qmv_ring_built(BITS, GS, STEPS, MR, 2))
      if (p.ring == 2) return qmv_tiles<BITS, GS, STEPS, MR, NMAT, 2>(a, p, st);
    return set_error(MLXQ_EINVAL, "qmv: no kernel with %d load rounds for this plan", p.ring);
  } else {
    return set_error(MLXQ_EINVAL, "qmv: %d load steps per wave with %d rows exceed the registers", STEPS, MR);
  }
}

template <int BITS, int GS, int STEPS, int NMAT>
static int qmv_rows(const QmvArgs& a, const QmvPlan& p, hipStream_t st) {
  switch (p.mr) {
    case 1: return qmv_mr<BITS, GS, STEPS, 1, NMAT>(a, p, st);
    case 2: return qmv_mr<BITS, GS, STEPS, 2, NMAT>(a, p, st);
    case 4: return qmv_mr<BITS, GS, STEPS, 4, NMAT>(a, p, st);
    default: return qmv_mr<BITS, GS, STEPS, 8, NMAT>(a, p, st);
  }
}

template <int BITS, int GS, int NMAT>
static int qmv_steps(const QmvArgs& a, const QmvPlan& p, hipStream_t st) {
  switch (p.steps) {
    case 1: return qmv_rows<BITS, GS, 1, NMAT>(a, p, st);
    case 2: return qmv_rows<BITS, GS, 2, NMAT>(a, p, st);
    case 3: return qmv_rows<BITS, GS, 3, NMAT>(a, p, st);
    case 4: return qmv_rows<BITS, GS, 4, NMAT>(a, p, st);
    case 6: return qmv_rows<BITS, GS, 6, NMAT>(a, p, st);
    default: return qmv_rows<BITS, GS, 8, NMAT>(a, p, st);
  }
}

// The tile kernels of one (bits, group size) pair; one translation unit each (qmv_tile_*.hip), so
// that they compile side by side.
#define MLXQ_QMV_TILE(BITS, GS)                                                              \
  int qmv_tile_##BITS##_##GS(const QmvArgs& a, const QmvPlan& p, int nmat, hipStream_t st) { \
    return nmat == 2 ? qmv_steps<BITS, GS, 2>(a, p, st) : qmv_steps<BITS, GS, 1>(a, p, st);  \
  }
int qmv_tile_4_32(const QmvArgs& a, const QmvPlan& p, int nmat, hipStream_t st);
int qmv_tile_4_64(const QmvArgs& a, const QmvPlan& p, int nmat, hipStream_t st);
int qmv_tile_4_128(const QmvArgs& a, const QmvPlan& p, int nmat, hipStream_t st);
int qmv_tile_8_32(const QmvArgs& a, const QmvPlan& p, int nmat, hipStream_t st);
int qmv_tile_8_64(const QmvArgs& a, const QmvPlan& p, int nmat, hipStream_t st);
int qmv_tile_8_128(const QmvArgs& a, const QmvPlan& p, int nmat, hipStream_t st);

}  // namespace mlxq
