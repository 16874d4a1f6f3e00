// qmv_mfma.hip — the decode GEMV's one-row kernel (M = 1, Q4) and the dispatch over it and the tile
// kernels of qmv_mfma.h.
#include "qmv_mfma.h"

namespace mlxq {

// ---------------------------------------------------------------------------------------------
// M = 1, Q4: one weight row per wave.
//
// A wave streams its whole row (its gate and up rows in the SwiGLU form) in contiguous 512-byte
// loads, 8 bytes per lane, all issued up front, and computes the row's dot product alone: no
// split-K partials, no reduction through LDS, and no workgroup barrier after the one that
// publishes the staged activations.  (Streaming rows whole measured 3.66-3.70 us for the down
// codes against 4.08 us for the 16-row x 64-byte loads of the tile kernel above.)
//
// A 512-byte load holds 16 columns of 64 codes.  Lane L reads bytes [32n + 8q, +8) with
// n = L & 15, q = L >> 4: codes [16q, 16q + 16) of column n, i.e. its two words feed two MFMAs
// (v_mfma_f32_16x16x32_bf16) whose B column n is column n's 64 codes.  The A operand's row m is
// the activation run of column m (16 different K slices of the one activation row), so the
// product's diagonal C[n][n] is column n's dot product sum x*c, and the off-diagonal
// entries are discarded.  A row of K codes takes LS = ceil(K / 1024) loads; when K is not a
// multiple of 1024 the last load's upper columns reach into the next row (or past the buffer end,
// where the loads return zero), and those columns fold exactly zero: their staged activations,
// activation sums and (s, b) table entries are all zero.  C[n][n] sits in lane n + 16 (n >> 2), register n & 3: 16 lanes of the
// wave fold one column each per load,
//   y += s*C[n][n] + b*X[column],
// with X the column's activation sum (computed once per workgroup while staging).  The wave's
// 16 partial sums are added at the end with row shifts and lane reads.
constexpr int kRowColPitch = 144;  // LDS bytes per 64-element activation column (128 + pad)

// Loads per row (K <= 1024 times this): 32 for one matrix, 16 for the SwiGLU pair, whose wave
// holds two rows' codes in registers.
constexpr int kRowMaxLoads[2] = {32, 16};

// Whether the one-row kernel takes a problem (bf16 x and scales are checked by the caller): the
// group count per row must be even (scales and biases are read as group pairs, 4-byte aligned).
__host__ __device__ constexpr bool qmv_row_fits(int64_t M, int64_t K, int gs, int bits, int nmat) {
  return M == 1 && bits == 4 && (gs == 64 || gs == 128) && K % (2 * gs) == 0 && K >= 1024 &&
         K <= 1024 * kRowMaxLoads[nmat - 1];
}

// LDS bytes of a one-row workgroup: the activation columns, their sums and each wave's (s, zc)
// table per matrix.
__host__ __device__ constexpr int qmv_row_lds(int LS, bool g64, int nmat, int wpb) {
  return LS * 16 * kRowColPitch + LS * 16 * 4 + wpb * nmat * (g64 ? LS * 16 : LS * 8) * 8;
}

template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}

// Contract (checked on the host by qmv_row_fits): M = 1, 1024 (LS - 1) < K <= 1024 LS, an even
// number of groups per row, bf16 x/scales/biases, Q4 codes, group 64 or 128, 8..16 waves per
// workgroup, dynamic LDS of qmv_row_lds bytes, every buffer < 2 GiB.  NMAT = 2: wave f streams
// gate row f and up row f and writes round(silu(round(g)) * round(u)) with
// silu(g) = round(g * round(sigmoid(g))) (qwen3.rs:178-181, src/nn.rs:301-303); else round(y).
// VALU: the same loads, unpack, staging and fold with the matrix cores left out — each lane forms
// the dot product of its 16 codes with their activations by v_dot2_f32_bf16, two products per
// instruction with f32 accumulation (y += s * dot, plus b * X once per column), and all 64 lanes' partial sums are added at the end.  It exists for the kernel-choice
// A/B (mlxq_qmv_valu), not for quantized_matmul.
template <bool G64, int LS, int NMAT, bool VALU>
__device__ __forceinline__ void qmv_row_body(
    const uint16_t* __restrict__ x, const uint32_t* __restrict__ wq, const uint16_t* __restrict__ scales,
    const uint16_t* __restrict__ biases, const uint32_t* __restrict__ wq2,
    const uint16_t* __restrict__ scales2, const uint16_t* __restrict__ biases2, int K, int N,
    uint16_t* __restrict__ y, const uint16_t* __restrict__ bias, const uint16_t* __restrict__ act_table) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  constexpr int C = 16 * LS;                  // 64-code columns per row, padded to whole loads
  constexpr int G = G64 ? C : C / 2;          // groups per padded row (table entries)
  constexpr int XCH = 128 * LS;               // 16-byte activation chunks of the padded row
  constexpr int XPT = (XCH + 511) / 512;      // ... per thread (at least 8 waves)
  constexpr int SBPL = (G + 127) / 128;       // scale/bias word pairs per lane
  const int Gr = K / (G64 ? 64 : 128);        // groups per row
  const uint32_t RB = (uint32_t)K / 2u;       // bytes per packed row
  const int NT = blockDim.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = blockIdx.x * (NT >> 6) + wave;
  const int r = row < N ? row : N - 1;  // waves past N take part in the staging, store nothing
  unsigned char* xs = lds;
  float* xsum = reinterpret_cast<float*>(lds + C * kRowColPitch);
  float* tab = xsum + C + wave * NMAT * G * 2;

  // Operand loads first (they queue ahead of the weight streams), then every weight load.  The
  // activation chunks past K read as zeros (past the resource's end).
  const auto rx = make_rsrc(x, K * 2);
  u32x4 cx[XPT];
#pragma unroll
  for (int j = 0; j < XPT; ++j) {
    const int ch = tid + j * NT;
    cx[j] = load16(rx, ch < XCH ? (uint32_t)ch * 16u : kOob);
  }
  const int sb_bytes = (int)((uint32_t)N * (uint32_t)Gr * 2u);
  uint32_t cs[NMAT][SBPL], cb[NMAT][SBPL];
#pragma unroll
  for (int mat = 0; mat < NMAT; ++mat) {
    const auto rs = make_rsrc(mat ? scales2 : scales, sb_bytes);
    const auto rz = make_rsrc(mat ? biases2 : biases, sb_bytes);
#pragma unroll
    for (int i = 0; i < SBPL; ++i) {
      const int g0 = 2 * lane + 128 * i;
      const uint32_t off = g0 < Gr ? ((uint32_t)r * (uint32_t)Gr + (uint32_t)g0) * 2u : kOob;
      cs[mat][i] = __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0);
      cb[mat][i] = __builtin_amdgcn_raw_buffer_load_b32(rz, off, 0, 0);
    }
  }
  // Every wave's activation loads go ahead of all weight streams in the CU's in-order memory
  // queue: the staging below needs the whole workgroup's (a bare s_barrier, no memory wait).
  __builtin_amdgcn_s_barrier();
  // Weight loads in fold order (step d of every matrix before step d + 1), so a step's operands
  // arrive together.
  u32x2 wv[NMAT][LS];
  const uint32_t lo = 32u * (uint32_t)(lane & 15) + 8u * (uint32_t)(lane >> 4);
  const int w_bytes = (int)((uint32_t)N * RB);
  const __amdgpu_buffer_rsrc_t rw[2] = {make_rsrc(wq, w_bytes), make_rsrc(NMAT == 2 ? wq2 : wq, w_bytes)};
#pragma unroll
  for (int d = 0; d < LS; ++d) {
#pragma unroll
    for (int mat = 0; mat < NMAT; ++mat)
      wv[mat][d] = __builtin_bit_cast(
          u32x2, __builtin_amdgcn_raw_buffer_load_b64(rw[mat], (uint32_t)r * RB + (uint32_t)d * 512u + lo, 0, 0));
  }

  // Activation columns (runs permuted to the unpacked code order) and their sums: the 8 chunks
  // of a column sit in 8 consecutive lanes of one wave (NT is a multiple of 64).
#pragma unroll
  for (int j = 0; j < XPT; ++j) {
    const int ch = tid + j * NT;
    const u32x4 v = cx[j];
    float t = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) t += __uint_as_float(v[e] << 16) + __uint_as_float(v[e] & 0xffff0000u);
    t += dpp_f32<0xb1>(t);   // quad_perm [1,0,3,2]
    t += dpp_f32<0x4e>(t);   // quad_perm [2,3,0,1]: every lane holds its quad's sum
    t += dpp_f32<0x104>(t);  // row_shl:4: lane 8k adds lane 8k+4's quad
    // (only lanes 8k, the column's first chunk, store the sum)
    if (ch < XCH) {
      *reinterpret_cast<u32x4*>(xs + (ch >> 3) * kRowColPitch + (ch & 7) * 16) = perm_q4(v);
      if ((ch & 7) == 0) xsum[ch >> 3] = t;
    }
  }
  // Publish the activations with LDS-only fences: a __syncthreads() release fence would also
  // wait for every outstanding weight load.
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  // The wave's (s, b) pairs per group, f32, after the barrier: only this wave reads them,
  // so the workgroup waits for the activations alone, not for every wave's scale loads.  Groups
  // past the row's end get (0, 0) (their loads returned zero).
#pragma unroll
  for (int mat = 0; mat < NMAT; ++mat) {
#pragma unroll
    for (int i = 0; i < SBPL; ++i) {
      const int g0 = 2 * lane + 128 * i;
      if (g0 < G) {
        const float s0 = __uint_as_float(cs[mat][i] << 16), s1 = __uint_as_float(cs[mat][i] & 0xffff0000u);
        const float b0 = __uint_as_float(cb[mat][i] << 16), b1 = __uint_as_float(cb[mat][i] & 0xffff0000u);
        *reinterpret_cast<f32x4*>(tab + (mat * G + g0) * 2) = f32x4{s0, b0, s1, b1};
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");

  // Load d covers columns 16d .. 16d+15.  Lane (m, q) = (L & 15, L >> 4) reads A runs 2q, 2q+1 of
  // column 16d + m, and folds column 16d + n (n = m) from register e = L & 3 of the product.
  const int m = lane & 15, q = lane >> 4, e = lane & 3;
  const unsigned char* xa = xs + m * kRowColPitch + q * 32;
  bf16x8 a[LS][2];
  f32x2 p[LS][NMAT];
  float xg[LS];
  f32x4 acc[LS][NMAT];
  float ya[NMAT];
#pragma unroll
  for (int mat = 0; mat < NMAT; ++mat) ya[mat] = 0.0f;
  auto read_step = [&](int d) {
    a[d][0] = *reinterpret_cast<const bf16x8*>(xa + d * 16 * kRowColPitch);
    a[d][1] = *reinterpret_cast<const bf16x8*>(xa + d * 16 * kRowColPitch + 16);
    const int col = 16 * d + m;
    const int g = G64 ? col : col >> 1;
#pragma unroll
    for (int mat = 0; mat < NMAT; ++mat) p[d][mat] = *reinterpret_cast<const f32x2*>(tab + (mat * G + g) * 2);
    xg[d] = xsum[col];
  };
  auto mfma_step = [&](int d) {
#pragma unroll
    for (int mat = 0; mat < NMAT; ++mat) {
      if constexpr (VALU) {
        // unpack_q4's pairs line up with the activation run's bf16 pairs (the MFMA operands'
        // element order), so each v_dot2 adds two code-activation products.
        float part[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const u32x4 wb = __builtin_bit_cast(u32x4, unpack_q4(wv[mat][d][h]));
          const u32x4 xr = __builtin_bit_cast(u32x4, a[d][h]);
          float t = 0.0f;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            // Elements copied out first: __builtin_bit_cast of a vector subscript (xr[j]) reads
            // element 0 for every j with this compiler.
            const uint32_t xj = xr[j], wj = wb[j];
            t = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, xj), __builtin_bit_cast(bf16x2, wj), t, false);
          }
          part[h] = t;
        }
        const float dot = part[0] + part[1];
        acc[d][mat][0] = dot;
      } else {
        const f32x4 c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[d][0], unpack_q4(wv[mat][d][0]),
                                                                f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
        acc[d][mat] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[d][1], unpack_q4(wv[mat][d][1]), c, 0, 0, 0);
      }
    }
  };
  auto fold_step = [&](int d) {
#pragma unroll
    for (int mat = 0; mat < NMAT; ++mat) {
      if constexpr (VALU) {
        // lane (m, q): s times its 16 codes' dot product; b times the column's activation sum
        // once per column (q == 0)
        ya[mat] = fmaf(p[d][mat][0], acc[d][mat][0], fmaf(q == 0 ? p[d][mat][1] : 0.0f, xg[d], ya[mat]));
      } else {
        const f32x4 c = acc[d][mat];
        float v = e == 1 ? c[1] : c[0];
        v = e == 2 ? c[2] : v;
        v = e == 3 ? c[3] : v;
        ya[mat] = fmaf(p[d][mat][0], v, fmaf(p[d][mat][1], xg[d], ya[mat]));
      }
      asm volatile("" : "+v"(ya[mat]));
    }
  };
  read_step(0);
#pragma unroll
  for (int d = 0; d < LS; ++d) {
    __builtin_amdgcn_sched_barrier(0);
    if (d + 1 < LS) read_step(d + 1 < LS ? d + 1 : d);
    mfma_step(d);
    if (d > 0) fold_step(d - 1);
  }
  __builtin_amdgcn_sched_barrier(0);
  fold_step(LS - 1);

  // The 16 diagonal lanes (n + 16 (n >> 2)) hold the partial sums (every lane in the VALU form):
  // a row-shift scan leaves each 16-lane row's sum in its lane 15.
  const bool diag = VALU || q == (m >> 2);
  float tot[NMAT];
#pragma unroll
  for (int mat = 0; mat < NMAT; ++mat) {
    float v = diag ? ya[mat] : 0.0f;
    v += dpp_f32<0x111>(v);
    v += dpp_f32<0x112>(v);
    v += dpp_f32<0x114>(v);
    v += dpp_f32<0x118>(v);
    tot[mat] = (__int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 15)) +
                __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 31))) +
               (__int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 47)) +
                __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63)));
  }
  if (lane == 0 && row < N) {
    const float v = tot[0];
    if constexpr (NMAT == 2) {
      // each op rounded to bf16 as the reference's separate ops are (qwen3.rs:178-181)
      y[row] = f32_to_bf16_bits(silu_bf16(round_bf16(v)) * round_bf16(tot[1]));
    } else {
      y[row] = gemv_finish(v, row, bias, act_table);
    }
  }
}

// Arguments in the order they are needed, a signature for each form, as the tile kernels have.
template <bool G64, int LS, bool VALU>
__global__ __launch_bounds__(1024) void qmv_row_kernel(
    const uint16_t* __restrict__ x, const uint32_t* __restrict__ wq, const uint16_t* __restrict__ scales,
    const uint16_t* __restrict__ biases, int K, int N, uint16_t* __restrict__ y, const uint16_t* __restrict__ bias,
    const uint16_t* __restrict__ act_table, QmmBatch bat) {
  // Stacked launch: the workgroup's y index selects the matrix (expert).
  if (const int64_t e = blockIdx.y; e > 0) {
    x += e * bat.x;
    wq += e * bat.w;
    scales += e * bat.sb;
    biases += e * bat.sb;
    y += e * bat.y;
    if (bias) bias += e * bat.bias;
  }
  qmv_row_body<G64, LS, 1, VALU>(x, wq, scales, biases, nullptr, nullptr, nullptr, K, N, y, bias, act_table);
}

template <bool G64, int LS>
__global__ __launch_bounds__(1024) void swiglu_row_kernel(
    const uint16_t* __restrict__ x, const uint32_t* __restrict__ wq, const uint16_t* __restrict__ scales,
    const uint16_t* __restrict__ biases, const uint32_t* __restrict__ wq2, const uint16_t* __restrict__ scales2,
    const uint16_t* __restrict__ biases2, int K, int N, uint16_t* __restrict__ y) {
  qmv_row_body<G64, LS, 2, false>(x, wq, scales, biases, wq2, scales2, biases2, K, N, y, nullptr, nullptr);
}

template <int NMAT>
static int qmv_kind(const QmvArgs& a, int gs, int bits, const QmvPlan& p, hipStream_t st) {
  if (bits == 8) {
    if (gs == 32) return qmv_tile_8_32(a, p, NMAT, st);
    if (gs == 64) return qmv_tile_8_64(a, p, NMAT, st);
    return qmv_tile_8_128(a, p, NMAT, st);
  }
  if (gs == 32) return qmv_tile_4_32(a, p, NMAT, st);
  if (gs == 64) return qmv_tile_4_64(a, p, NMAT, st);
  return qmv_tile_4_128(a, p, NMAT, st);
}

// CUs of the current device.
static int64_t gemv_cus() { return device_cu_count(); }

// Waves (rows) per one-row workgroup.  SwiGLU (two rows per wave): 8, i.e. the staging barrier
// among fewer waves (K = 3072, F = 8192: 7.7 -> 7.1 us against 16 waves; 4 measured slower).
// One matrix: of 16, 12 and 8 the one whose busiest CU streams the fewest rows,
// ceil(ceil(N / w) / CUs) * w, the larger on a tie.  Measured over 14 shapes (K = 2048..28672,
// N = 1536..8192) the launch time follows that count: N = 3072 takes 12 (4.74 us against 4.94 at 8
// and 5.37 at 16), N = 5120 takes 12 (K = 13824: 13.6 us against 15.1 at 16), N = 1536 takes 8
// (3.99 against 5.29 at 16), N = 3584 and 8192 take 16.
static int qmv_row_wpb(int64_t N, int nmat) {
  if (nmat == 2) return 8;
  const int64_t cus = gemv_cus();
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

template <bool G64, int LS, int NMAT, bool VALU = false>
static int launch_qmv_row(const QmvArgs& a, hipStream_t st) {
  static_assert(qmv_row_lds(LS, G64, NMAT, 16) <= kMaxLds, "one-row workgroup exceeds the LDS");
  static std::atomic<bool> attr_set[64];
  const void* kernel;
  if constexpr (NMAT == 1) kernel = reinterpret_cast<const void*>(&qmv_row_kernel<G64, LS, VALU>);
  else kernel = reinterpret_cast<const void*>(&swiglu_row_kernel<G64, LS>);
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return set_error(MLXQ_EDEVICE, "qmv: no current device");
  if (dev < 0 || dev >= 64 || !attr_set[dev].load(std::memory_order_acquire)) {
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds) != hipSuccess)
      return set_error(MLXQ_EDEVICE, "qmv: hipFuncSetAttribute failed");
    if (dev >= 0 && dev < 64) attr_set[dev].store(true, std::memory_order_release);
  }
  const int wpb = qmv_row_wpb(a.N, NMAT);
  const int lds = qmv_row_lds(LS, G64, NMAT, wpb);
  const dim3 grid((unsigned)((a.N + wpb - 1) / wpb), (unsigned)a.bat.count), block(wpb * 64);
  if constexpr (NMAT == 1)
    hipLaunchKernelGGL((qmv_row_kernel<G64, LS, VALU>), grid, block, lds, st, (const uint16_t*)a.x, a.wq, (const uint16_t*)a.s,
                       (const uint16_t*)a.b, (int)a.K, (int)a.N, (uint16_t*)a.y, a.bias, a.act_table, a.bat);
  else
    hipLaunchKernelGGL((swiglu_row_kernel<G64, LS>), grid, block, lds, st, (const uint16_t*)a.x, a.wq, (const uint16_t*)a.s,
                       (const uint16_t*)a.b, a.wq2, (const uint16_t*)a.s2, (const uint16_t*)a.b2, (int)a.K, (int)a.N,
                       (uint16_t*)a.y);
  return check_launch(NMAT == 2 ? "swiglu_qmv_row" : VALU ? "qmv_row_valu" : "qmv_row");
}

// Launchers by loads per row (1 .. kRowMaxLoads).
template <bool G64, int NMAT, bool VALU = false, int... L>
static int qmv_row_ls(const QmvArgs& a, hipStream_t st, std::integer_sequence<int, L...>) {
  using Launch = int (*)(const QmvArgs&, hipStream_t);
  static constexpr Launch launch[] = {&launch_qmv_row<G64, L + 1, NMAT, VALU>...};
  return launch[(a.K + 1023) / 1024 - 1](a, st);
}

template <int NMAT>
static int qmv_row(const QmvArgs& a, int gs, hipStream_t st) {
  constexpr auto ls = std::make_integer_sequence<int, kRowMaxLoads[NMAT - 1]>{};
  return gs == 64 ? qmv_row_ls<true, NMAT>(a, st, ls) : qmv_row_ls<false, NMAT>(a, st, ls);
}

static bool buffers_fit(int64_t M, int64_t K, int64_t N) {
  const int64_t lim = (int64_t)1 << 31;  // every buffer (Q8 weights: N*K bytes) under 2 GiB
  return N * K < lim && M * K * 2 < lim;
}

bool qmv_mfma_applicable(int x_dtype, int sb_dtype, int64_t M, int64_t K, int64_t N, int gs, int bits) {
  if (x_dtype != MLXQ_BFLOAT16 || sb_dtype != MLXQ_BFLOAT16 || !buffers_fit(M, K, N)) return false;
  QmvPlan p;
  return qmv_row_fits(M, K, gs, bits, 1) || qmv_plan(M, K, gs, bits, 1, p);
}

int run_qmv_mfma(const void* x, int64_t M, int64_t K, const uint32_t* wq, const void* s, const void* b,
                 int64_t N, int gs, int bits, void* y, hipStream_t st, const uint16_t* bias, const uint16_t* act_table,
                 const QmmBatch& bat) {
  const QmvArgs a = {x, M, K, N, wq, s, b, nullptr, nullptr, nullptr, y, bias, act_table, bat};
  if (qmv_row_fits(M, K, gs, bits, 1)) return qmv_row<1>(a, gs, st);
  QmvPlan p;
  if (!qmv_plan(M, K, gs, bits, 1, p))
    return set_error(MLXQ_EINVAL, "qmv: no GEMV plan for M=%lld K=%lld", (long long)M, (long long)K);
  if (p.rows == M) return qmv_kind<1>(a, gs, bits, p, st);
  for (int64_t m0 = 0; m0 < M; m0 += p.rows) {  // launches of p.rows activation rows
    const int64_t rows = M - m0 < p.rows ? M - m0 : p.rows;
    const int rc = run_qmv_mfma(static_cast<const uint16_t*>(x) + m0 * K, rows, K, wq, s, b, N, gs, bits,
                                static_cast<uint16_t*>(y) + m0 * N, st, bias, act_table, bat);
    if (rc != MLXQ_OK) return rc;
  }
  return MLXQ_OK;
}

// The VALU form of the one-row kernel (the kernel-choice A/B behind mlxq_qmv_valu): bf16 x and
// scales, M = 1, Q4 group 64/128, K up to kRowValuMaxLoads * 1024 (the decode shapes).
constexpr int kRowValuMaxLoads = 8;

bool qmv_row_valu_applicable(int x_dtype, int sb_dtype, int64_t M, int64_t K, int64_t N, int gs, int bits) {
  return x_dtype == MLXQ_BFLOAT16 && sb_dtype == MLXQ_BFLOAT16 && buffers_fit(M, K, N) &&
         qmv_row_fits(M, K, gs, bits, 1) && K <= 1024 * kRowValuMaxLoads;
}

int run_qmv_row_valu(const void* x, int64_t K, const uint32_t* wq, const void* s, const void* b, int64_t N,
                     int gs, void* y, hipStream_t st) {
  const QmvArgs a = {x, 1, K, N, wq, s, b, nullptr, nullptr, nullptr, y};
  constexpr auto ls = std::make_integer_sequence<int, kRowValuMaxLoads>{};
  return gs == 64 ? qmv_row_ls<true, 1, true>(a, st, ls) : qmv_row_ls<false, 1, true>(a, st, ls);
}

bool swiglu_qmv_applicable(int x_dtype, int sb_dtype, int64_t M, int64_t K, int64_t F, int gs, int bits) {
  if (x_dtype != MLXQ_BFLOAT16 || sb_dtype != MLXQ_BFLOAT16 || !buffers_fit(M, K, F)) return false;
  if (bits != 4 && bits != 8) return false;
  if (K % (512 / bits) != 0) return false;  // the fused form's stated condition
  QmvPlan p;
  return qmv_row_fits(M, K, gs, bits, 2) || qmv_plan(M, K, gs, bits, 2, p);
}

int run_swiglu_qmv(const void* x, int64_t M, int64_t K, const uint32_t* wq_g, const void* s_g,
                   const void* b_g, const uint32_t* wq_u, const void* s_u, const void* b_u, int64_t F,
                   int gs, int bits, void* h, hipStream_t st) {
  const QmvArgs a = {x, M, K, F, wq_g, s_g, b_g, wq_u, s_u, b_u, h};
  if (qmv_row_fits(M, K, gs, bits, 2)) return qmv_row<2>(a, gs, st);
  QmvPlan p;
  if (!qmv_plan(M, K, gs, bits, 2, p))
    return set_error(MLXQ_EUNSUPPORTED, "swiglu: no fused GEMV plan for M=%lld K=%lld", (long long)M,
                     (long long)K);
  if (p.rows == M) return qmv_kind<2>(a, gs, bits, p, st);
  for (int64_t m0 = 0; m0 < M; m0 += p.rows) {  // launches of p.rows activation rows
    const int64_t rows = M - m0 < p.rows ? M - m0 : p.rows;
    const int rc = run_swiglu_qmv(static_cast<const uint16_t*>(x) + m0 * K, rows, K, wq_g, s_g, b_g, wq_u, s_u,
                                  b_u, F, gs, bits, static_cast<uint16_t*>(h) + m0 * F, st);
    if (rc != MLXQ_OK) return rc;
  }
  return MLXQ_OK;
}

}  // namespace mlxq
