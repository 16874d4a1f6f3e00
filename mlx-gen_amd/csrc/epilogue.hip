// epilogue.hip — LoRA prologue and the unfused linear epilogue.
//
// The adapter residual of the reference (Adapter::residual: scale * (x.A).B, each matmul and the
// scale multiply rounded to the activation dtype) needs x.A once per call.  lora_prep computes it
// together with the transposed, zero-padded up-projection so the GEMM epilogue can run the
// rank-R product as one more MFMA K-step.  linear_epilogue applies bias / LoRA / activation to an
// already computed y for the paths that do not fuse them (GEMV, f32 activations, ranks above 16,
// further adapters and every result MLX's dtype promotion makes f32 from a bf16 product).
#include "mlxq_common.h"

namespace mlxq {

// xa[M,R] = round(x[M,K] . A[K,rank]) (zero for r >= rank); lbt[N,R] = B[rank,N]^T (zero padded).
// One thread per output element: the general form (f32 activations, K not a multiple of 32).
template <typename XT>
__global__ void lora_prep_kernel(const XT* __restrict__ x, int64_t M, int64_t K,
                                 const XT* __restrict__ A, const XT* __restrict__ B, int64_t N,
                                 int rank, int R, XT* __restrict__ xa, XT* __restrict__ lbt) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nxa = M * R;
  if (t < nxa) {
    const int64_t m = t / R;
    const int r = (int)(t % R);
    float acc = 0.0f;
    if (r < rank) {
      for (int64_t k = 0; k < K; ++k) acc = fmaf(Act<XT>::ld(x, m * K + k), Act<XT>::ld(A, k * rank + r), acc);
    }
    Act<XT>::st(xa, t, acc);
  } else if (t < nxa + N * R) {
    const int64_t u = t - nxa;
    const int64_t n = u / R;
    const int r = (int)(u % R);
    lbt[u] = r < rank ? B[(int64_t)r * N + n] : (XT)0;
  }
}

// bf16 x.A on the matrix cores: xa[M,R] = round_bf16(x[M,K] . A[K,rank]), columns >= rank zero.
// A workgroup owns `rows` rows of x (NB blocks of 16 rows on the MFMA; rows past its share repeat
// its last row and are not stored) and 16 columns of xa; its 8 waves split K (32 per MFMA step,
// K % 32 == 0 because K is a multiple of the group size) and reduce through LDS.  The MFMA's B
// operand needs 8 consecutive k of one column of the k-major A: 8 two-byte loads per lane and
// step, L1/L2 hits (A is at most K x 256 x 2 bytes and every workgroup reads it).  Each wave
// walks its K range in chunks of kXaChunk steps, double-buffered: a chunk's loads are issued
// before the previous chunk's MFMAs, so a wave waits for memory about once instead of once per
// step (the x rows come from HBM).
constexpr int kXaWaves = 8;
constexpr int kXaChunk = 4;
// Workgroups past the x.A grid (blockIdx.x >= xa_blocks) write lbt[N,R] = B[rank,N]^T instead
// (zero padded, the GEMM epilogue's operand), so the LoRA preparation is one launch.
// A16 (rank 16, one 16-column block): a chunk of A (4 steps x 32 rows x 16 columns) is 4 KB of
// contiguous memory, fetched with four 16-byte loads per lane and transposed through the wave's
// 4 KB LDS buffer, instead of 32 two-byte gathers per lane.
// Rows per workgroup: 16, except from 4097 to 8192 rows, where ceil(M / 256) (17-32 rows, two
// MFMA blocks) spreads the x stream evenly over at most 256 workgroups, one per CU.  With 16-row
// workgroups M = 4608 made 288 of them, and the 32 CUs that ran two read twice the bytes: same-
// process A/B through mlxq_lora_residual (K = 3072, rank 16), 16-row against balanced workgroups:
// M = 4608 24.0 -> 20.9 us, 5120 23.8 -> 21.3, 6144 26.0 -> 24.3, 8192 29.9 / 30.1 (even);
// 512 balanced workgroups of up to 16 rows (two per CU) gained about half as much, and 32-row
// workgroups past 8192 rows lost (M = 12288 51.5 -> 53.1).
template <bool A16, int NB>
__global__ __launch_bounds__(kXaWaves * 64) void lora_xa_kernel(const uint16_t* __restrict__ x, int M,
                                                                int K, const uint16_t* __restrict__ A,
                                                                int rank, int R, uint16_t* __restrict__ xa,
                                                                int xa_blocks, int rows,
                                                                const uint16_t* __restrict__ B,
                                                                int64_t N, uint16_t* __restrict__ lbt) {
  __shared__ float red[NB][kXaWaves][16 * 16];
  __shared__ __attribute__((aligned(16))) uint16_t abuf[A16 ? kXaWaves * 2048 : 8];
  // wave is made scalar so the K-range branches below are uniform scalar branches.
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if ((int)blockIdx.x >= xa_blocks) {
    if (blockIdx.y != 0) return;
    const int64_t u = ((int64_t)blockIdx.x - xa_blocks) * (kXaWaves * 64) + tid;
    if (u < N * R) {
      const int64_t n = u / R;
      const int rr = (int)(u % R);
      lbt[u] = rr < rank ? B[(int64_t)rr * N + n] : (uint16_t)0;
    }
    return;
  }
  const int c16 = lane & 15, q = lane >> 4;
  const int m0 = blockIdx.x * rows, r0 = blockIdx.y * 16;
  const int m_end = m0 + rows < M ? m0 + rows : M;  // this workgroup's rows [m0, m_end)
  const int r = r0 + c16;
  const bool rvalid = r < rank;
  const int KS = K / 32, per = (KS + kXaWaves - 1) / kXaWaves;
  const int ks0 = __builtin_amdgcn_readfirstlane(wave * per);
  const int ks1 = __builtin_amdgcn_readfirstlane(ks0 + per < KS ? ks0 + per : KS);
  const uint16_t* xp[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int row = m0 + 16 * b + c16;
    xp[b] = x + (int64_t)(row < m_end ? row : m_end - 1) * K + 8 * q;
  }
  const uint16_t* ap = A + (int64_t)(8 * q) * rank + (rvalid ? r : 0);
  struct Chunk {
    bf16x8 a[NB][kXaChunk];
    uint16_t w[A16 ? 1 : kXaChunk][8];
    u32x4 araw[A16 ? kXaChunk : 1];  // A16: lane l's 64 bytes of the chunk (rows 2l, 2l+1)
  };
  uint16_t* const wbuf = abuf + (A16 ? wave * 2048 : 0);
  // Steps past the wave's range repeat its last step (in bounds) and are not accumulated.  Every
  // load is unconditional (lanes of columns >= rank read column 0 and zero it afterwards): a
  // conditional load made the compiler wait for each one before the next.
  auto load = [&](int ks, Chunk& c) {
#pragma unroll
    for (int u = 0; u < kXaChunk; ++u) {
      const int k = ks + u < ks1 ? ks + u : ks1 - 1;
#pragma unroll
      for (int b = 0; b < NB; ++b) c.a[b][u] = *reinterpret_cast<const bf16x8*>(xp[b] + k * 32);
      if constexpr (!A16) {
#pragma unroll
        for (int j = 0; j < 8; ++j) c.w[u][j] = ap[(int64_t)(k * 32 + j) * rank];  // column 0 if !rvalid
      }
    }
    if constexpr (A16) {
#pragma unroll
      for (int p = 0; p < kXaChunk; ++p) {  // row ks*32 + 2 lane + p/2, columns 8 (p&1) .. +8
        const int row = ks * 32 + 2 * lane + (p >> 1);
        c.araw[p] = *reinterpret_cast<const u32x4*>(A + (int64_t)(row < K ? row : K - 1) * 16 + 8 * (p & 1));
      }
    }
  };
  // A16: the chunk's rows into the wave's buffer, [128 rows][16 columns] bf16 (after this wave's
  // reads of the previous chunk, LDS being in order within a wave).
  auto stage = [&](const Chunk& c) {
    if constexpr (A16) {
#pragma unroll
      for (int p = 0; p < kXaChunk; ++p) *reinterpret_cast<u32x4*>(wbuf + lane * 32 + p * 8) = c.araw[p];
    }
  };
  f32x4 acc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // Every MFMA of a chunk is issued; steps past the wave's range and padding columns get a zero B
  // operand through a mask the compiler cannot see through.  MFMA does not honour the EXEC mask:
  // given a visible "operand is zero" condition the compiler predicated the MFMA on EXEC without
  // a branch, and with one step per wave it then added the repeated step a second time.
  auto compute = [&](int ks, const Chunk& c) {
#pragma unroll
    for (int u = 0; u < kXaChunk; ++u) {
      uint32_t keep = rvalid && ks + u < ks1 ? 0xffffffffu : 0u;
      asm volatile("" : "+v"(keep));
      u32x4 bw;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t lo, hi;
        if constexpr (A16) {
          lo = wbuf[(u * 32 + 8 * q + 2 * j) * 16 + c16];
          hi = wbuf[(u * 32 + 8 * q + 2 * j + 1) * 16 + c16];
        } else {
          lo = c.w[u][2 * j];
          hi = c.w[u][2 * j + 1];
        }
        bw[j] = (lo | (hi << 16)) & keep;
      }
#pragma unroll
      for (int b = 0; b < NB; ++b)
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c.a[b][u], __builtin_bit_cast(bf16x8, bw), acc[b], 0, 0, 0);
    }
  };
  if (ks0 < ks1) {
    Chunk c0, c1;
    load(ks0, c0);
    for (int ks = ks0; ks < ks1; ks += 2 * kXaChunk) {
      load(ks + kXaChunk, c1);
      stage(c0);
      compute(ks, c0);
      if (ks + kXaChunk < ks1) {
        load(ks + 2 * kXaChunk, c0);
        stage(c1);
        compute(ks + kXaChunk, c1);
      }
    }
  }
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e) red[b][wave][(4 * q + e) * 16 + c16] = acc[b][e];
  __syncthreads();
  if (tid < 256 * NB) {
    const int b = tid >> 8, m = (tid >> 4) & 15, n = tid & 15;
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < kXaWaves; ++w) v += red[b][w][m * 16 + n];
    const int row = m0 + 16 * b + m;
    if (row < m_end) xa[(int64_t)row * R + r0 + n] = f32_to_bf16_bits(v);
  }
}

// DR = f32 (an f32 or fp16 activation, or f32 factors): xa[M,R] = x . A and lbt[N,R] = B^T in f32,
// x and the factors widened exactly (MLX promotes the 16-bit operands of a mixed matmul to f32).
// One thread per output element: the general form (K not a multiple of 16, unaligned x).
template <typename XT, typename FT>
__global__ void lora_prep_f32_kernel(const XT* __restrict__ x, int64_t M, int64_t K,
                                     const FT* __restrict__ A, const FT* __restrict__ B, int64_t N,
                                     int rank, int R, float* __restrict__ xa, float* __restrict__ lbt) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nxa = M * R;
  if (t < nxa) {
    const int64_t m = t / R;
    const int r = (int)(t % R);
    float acc = 0.0f;
    if (r < rank) {
      for (int64_t k = 0; k < K; ++k) acc = fmaf(Act<XT>::ld(x, m * K + k), Act<FT>::ld(A, k * rank + r), acc);
    }
    xa[t] = acc;
  } else if (t < nxa + N * R) {
    const int64_t u = t - nxa;
    const int64_t n = u / R;
    const int r = (int)(u % R);
    lbt[u] = r < rank ? Act<FT>::ld(B, (int64_t)r * N + n) : 0.0f;
  }
}

// The same on v_mfma_f32_16x16x4_f32, whose products and sums are f32's own.  A workgroup owns 16
// rows of x and 16 * NCB columns of xa; its 8 waves split K and reduce through LDS.  Bound by the
// x stream and by the loads of A: per 16 k, a lane loads 4 consecutive x values of its row and, for
// each of those 4 k, the NCB adjacent columns (16 columns x NCB) of A its column index owns, so
// MFMA t multiplies k = 4 q + t of both sides with no transpose, and NCB = 2 or 4 (rank a multiple
// of it, A aligned to the wider load) halves or quarters both the loads of A and the passes over x.
// One thread per output, walking K alone, had taken 576 us for x [4608, 3072] f32, rank 32, where
// x's bytes take 11.5 us at copy speed; with lora_epilogue_kernel below, the whole linear
// [4608, 3072] x [12288, 3072]^T with rank 32 and GELU went from 7196 to 1043 us.
// Workgroups past xa_blocks write lbt, eight ranks of one n per thread (loads coalesced over n).
template <typename XT, typename FT, int NCB>
__global__ __launch_bounds__(kXaWaves * 64) void lora_xa_f32_kernel(
    const XT* __restrict__ x, int64_t M, int64_t K, const FT* __restrict__ A, const FT* __restrict__ B,
    int64_t N, int rank, int R, float* __restrict__ xa, float* __restrict__ lbt, int xa_blocks) {
  __shared__ float red[NCB][kXaWaves][16 * 16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if ((int)blockIdx.x >= xa_blocks) {
    if (blockIdx.y != 0) return;
    const int64_t u = ((int64_t)blockIdx.x - xa_blocks) * (kXaWaves * 64) + tid;
    if (u < N * (R / 8)) {
      const int64_t n = u % N;
      const int r8 = (int)(u / N) * 8;
      f32x4 v[2];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j >> 2][j & 3] = r8 + j < rank ? Act<FT>::ld(B, (int64_t)(r8 + j) * N + n) : 0.0f;
#pragma unroll
      for (int h = 0; h < 2; ++h) *reinterpret_cast<f32x4*>(lbt + n * R + r8 + 4 * h) = v[h];
    }
    return;
  }
  constexpr int U = NCB == 4 ? 2 : 4;  // 16-deep steps per chunk, double-buffered
  struct alignas(4 * sizeof(XT)) XV { XT v[4]; };
  struct alignas(NCB * sizeof(FT)) AV { FT v[NCB]; };
  struct Chunk {
    XV x[U];
    AV a[U][4];
  };
  const int c16 = lane & 15, q = lane >> 4;
  const int64_t m0 = (int64_t)blockIdx.x * 16;
  const int r0 = blockIdx.y * 16 * NCB;
  const int col = r0 + c16 * NCB;  // this lane's first column; rank is a multiple of NCB
  const int KS = (int)(K / 16);
  const int ks0 = __builtin_amdgcn_readfirstlane((int)((int64_t)wave * KS / kXaWaves));
  const int ks1 = __builtin_amdgcn_readfirstlane((int)((int64_t)(wave + 1) * KS / kXaWaves));
  const XT* xp = x + (m0 + c16 < M ? m0 + c16 : M - 1) * K + 4 * q;
  const FT* ap = A + (int64_t)(4 * q) * rank + (col < rank ? col : 0);  // padding columns: not stored
  auto load1 = [&](int ks, XV& xv, AV (&av)[4]) {
    xv = *reinterpret_cast<const XV*>(xp + (int64_t)ks * 16);
#pragma unroll
    for (int t = 0; t < 4; ++t) av[t] = *reinterpret_cast<const AV*>(ap + ((int64_t)ks * 16 + t) * rank);
  };
  f32x4 acc[NCB];
#pragma unroll
  for (int c = 0; c < NCB; ++c) acc[c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto mac1 = [&](const XV& xv, const AV (&av)[4]) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int c = 0; c < NCB; ++c)
        acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(Act<XT>::ld(xv.v, t), Act<FT>::ld(av[t].v, c), acc[c], 0, 0, 0);
  };
  auto load = [&](int ks, Chunk& c) {
#pragma unroll
    for (int u = 0; u < U; ++u) load1(ks + u, c.x[u], c.a[u]);
  };
  auto mac = [&](const Chunk& c) {
#pragma unroll
    for (int u = 0; u < U; ++u) mac1(c.x[u], c.a[u]);
  };
  // Whole chunks, the next one's loads ahead of this one's products, then single steps; every
  // condition is wave-uniform.
  const int full = (ks1 - ks0) / U;
  if (full > 0) {
    Chunk c0, c1;
    load(ks0, c0);
    for (int i = 0; i < full; i += 2) {
      if (i + 1 < full) load(ks0 + (i + 1) * U, c1);
      mac(c0);
      if (i + 1 < full) {
        if (i + 2 < full) load(ks0 + (i + 2) * U, c0);
        mac(c1);
      }
    }
  }
  for (int ks = ks0 + full * U; ks < ks1; ++ks) {
    XV xv;
    AV av[4];
    load1(ks, xv, av);
    mac1(xv, av);
  }
#pragma unroll
  for (int c = 0; c < NCB; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) red[c][wave][(4 * q + e) * 16 + c16] = acc[c][e];
  __syncthreads();
  for (int i = tid; i < 256 * NCB; i += kXaWaves * 64) {
    const int m = i / (16 * NCB), cc = i % (16 * NCB);  // cc: column r0 + cc = block cc % NCB, index cc / NCB
    float v = 0.0f;
#pragma unroll
    for (int w = 0; w < kXaWaves; ++w) v += red[cc % NCB][w][m * 16 + cc / NCB];
    if (m0 + m < M && r0 + cc < R) xa[(m0 + m) * R + r0 + cc] = r0 + cc < rank ? v : 0.0f;
  }
}

template <typename XT, typename FT>
static int lora_prep_f32(const void* x, int64_t M, int64_t K, const void* A, const void* B, int64_t N, int rank,
                         int R, void* xa, void* lbt, hipStream_t st) {
  const auto aligned = [](const void* p, size_t a) { return reinterpret_cast<uintptr_t>(p) % a == 0; };
  const int64_t xa_blocks = (M + 15) / 16, bt_blocks = (N * (R / 8) + kXaWaves * 64 - 1) / (kXaWaves * 64);
  if (K % 16 == 0 && aligned(x, 4 * sizeof(XT)) && K < (1LL << 31) && xa_blocks + bt_blocks < (1LL << 31)) {
#define MLXQ_XA(C)                                                                                               \
  hipLaunchKernelGGL((lora_xa_f32_kernel<XT, FT, C>), dim3((unsigned)(xa_blocks + bt_blocks), (unsigned)((R + 16 * C - 1) / (16 * C))), \
                     dim3(kXaWaves * 64), 0, st, (const XT*)x, M, K, (const FT*)A, (const FT*)B, N, rank, R,     \
                     (float*)xa, (float*)lbt, (int)xa_blocks)
    if (R > 32 && rank % 4 == 0 && aligned(A, 4 * sizeof(FT))) MLXQ_XA(4);
    else if (R > 16 && rank % 2 == 0 && aligned(A, 2 * sizeof(FT))) MLXQ_XA(2);
    else MLXQ_XA(1);
#undef MLXQ_XA
    return check_launch("lora_prep");
  }
  const int64_t blocks = (M * R + N * R + 255) / 256;
  if (blocks > 0x7fffffff) return set_error(MLXQ_EINVAL, "lora: problem too large");
  hipLaunchKernelGGL((lora_prep_f32_kernel<XT, FT>), dim3((unsigned)blocks), dim3(256), 0, st, (const XT*)x, M, K,
                     (const FT*)A, (const FT*)B, N, rank, R, (float*)xa, (float*)lbt);
  return check_launch("lora_prep");
}

int run_lora_prep(const void* x, int x_dtype, int64_t M, int64_t K, const void* A, const void* B,
                  int lora_dtype, int64_t N, int rank, int R, void* xa, void* lbt, hipStream_t st) {
  const int64_t total = M * R + N * R;
  if (total == 0) return MLXQ_OK;
  const int64_t blocks = (total + 255) / 256;
  if (blocks > 0x7fffffff) return set_error(MLXQ_EINVAL, "lora: problem too large");
  if (x_dtype != MLXQ_BFLOAT16 || lora_dtype != MLXQ_BFLOAT16) {
    const bool fb = lora_dtype == MLXQ_BFLOAT16;
    if (x_dtype == MLXQ_FLOAT16)
      return fb ? lora_prep_f32<_Float16, uint16_t>(x, M, K, A, B, N, rank, R, xa, lbt, st)
                : lora_prep_f32<_Float16, float>(x, M, K, A, B, N, rank, R, xa, lbt, st);
    if (x_dtype == MLXQ_BFLOAT16) return lora_prep_f32<uint16_t, float>(x, M, K, A, B, N, rank, R, xa, lbt, st);
    return fb ? lora_prep_f32<float, uint16_t>(x, M, K, A, B, N, rank, R, xa, lbt, st)
              : lora_prep_f32<float, float>(x, M, K, A, B, N, rank, R, xa, lbt, st);
  }
  const int64_t bt_blocks = (N * R + kXaWaves * 64 - 1) / (kXaWaves * 64);
  if (K % 32 == 0 && M < (1LL << 31) / 16 && K < (1LL << 31) && bt_blocks < (1LL << 30)) {
    // x.A workgroups (`rows` rows x 16 columns each), then the B^T workgroups.
    const int rows = M > 16 * 256 && M <= 32 * 256 ? (int)((M + 255) / 256) : 16;
    const int xa_blocks = (int)((M + rows - 1) / rows);
    const dim3 grid((unsigned)(xa_blocks + bt_blocks), (unsigned)(R / 16));
    if (rows <= 16) {
      if (rank == 16 && R == 16)
        hipLaunchKernelGGL((lora_xa_kernel<true, 1>), grid, dim3(kXaWaves * 64), 0, st, (const uint16_t*)x,
                           (int)M, (int)K, (const uint16_t*)A, rank, R, (uint16_t*)xa, xa_blocks, rows,
                           (const uint16_t*)B, N, (uint16_t*)lbt);
      else
        hipLaunchKernelGGL((lora_xa_kernel<false, 1>), grid, dim3(kXaWaves * 64), 0, st, (const uint16_t*)x,
                           (int)M, (int)K, (const uint16_t*)A, rank, R, (uint16_t*)xa, xa_blocks, rows,
                           (const uint16_t*)B, N, (uint16_t*)lbt);
    } else {
      if (rank == 16 && R == 16)
        hipLaunchKernelGGL((lora_xa_kernel<true, 2>), grid, dim3(kXaWaves * 64), 0, st, (const uint16_t*)x,
                           (int)M, (int)K, (const uint16_t*)A, rank, R, (uint16_t*)xa, xa_blocks, rows,
                           (const uint16_t*)B, N, (uint16_t*)lbt);
      else
        hipLaunchKernelGGL((lora_xa_kernel<false, 2>), grid, dim3(kXaWaves * 64), 0, st, (const uint16_t*)x,
                           (int)M, (int)K, (const uint16_t*)A, rank, R, (uint16_t*)xa, xa_blocks, rows,
                           (const uint16_t*)B, N, (uint16_t*)lbt);
    }
  } else {
    hipLaunchKernelGGL(lora_prep_kernel<uint16_t>, dim3((unsigned)blocks), dim3(256), 0, st,
                       (const uint16_t*)x, M, K, (const uint16_t*)A, (const uint16_t*)B, N, rank, R,
                       (uint16_t*)xa, (uint16_t*)lbt);
  }
  return check_launch("lora_prep");
}

__device__ __forceinline__ float ld_any(const void* p, bool bf16, int64_t i) {
  return bf16 ? bf16_bits_to_f32(static_cast<const uint16_t*>(p)[i]) : static_cast<const float*>(p)[i];
}
__device__ __forceinline__ float rnd_if(bool bf16, float v) { return bf16 ? round_bf16(v) : v; }

// out = act(y1 + r), y1 = y_in + bias: every stage rounded to its promoted dtype (flags), the
// sequence of LinearBase::forward's bias add and AdaptableLinear::forward's residual sum
// (reference src/adapters.rs:318-320,543-549, Adapter::residual :260-270).  A bf16 activation is
// the bf16 table's entry of its input; in f32 it is evaluated (GELU and the exact GELU as the
// f32 erf form, the tanh GELU op by op).  has_r: r is the residual's product, before rounding.
__device__ __forceinline__ float epilogue_finish(const LinearEpilogueArgs& a, float o, int64_t n, bool has_r, float r) {
  if (a.bias) o = rnd_if(a.d1_bf16, o + ld_any(a.bias, a.bias_bf16, n));
  if (has_r) o = rnd_if(a.d2_bf16, o + rnd_if(a.dr_bf16, rnd_if(a.dr_bf16, r) * a.lora_scale));
  const bool act_bf16 = a.d2_bf16;  // the activation's input dtype
  if (a.act == MLXQ_ACT_GELU) {
    o = gelu_erf(o);
  } else if (a.act == MLXQ_ACT_GELU_TANH || a.act == MLXQ_ACT_GELU_EXACT) {
    if (act_bf16) o = bf16_bits_to_f32(a.act_table[f32_to_bf16_bits(o)]);
    else o = a.act == MLXQ_ACT_GELU_TANH ? gelu_tanh<false>(o) : gelu_erf(o);
  }
  return o;
}

// Without LoRA (R == 0): one thread per output.
template <typename YI, typename YO>
__global__ void linear_epilogue_kernel(LinearEpilogueArgs a) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= a.M * a.N) return;
  const float o = Act<YI>::ld(static_cast<const YI*>(a.y_in), t);
  Act<YO>::st(static_cast<YO*>(a.y_out), t, epilogue_finish(a, o, t % a.N, a.res != nullptr, a.res ? a.res[t] : 0.0f));
}

// With LoRA (R > 0): r = xa . lbt^T on the matrix cores (bf16 operands for DR = bf16, f32 operands
// for DR = f32, the products and sums f32's own), one 32 x 64 block of outputs per wave.  Meant to
// run at the rate of reading y_in and writing y_out; one thread per output, reading 2 R operands
// for each, had taken 5.7 ms for [4608, 12288] f32 at R = 32, where y's 453 MB take 92 us.  The
// activation rows are the MFMA's A side, so a lane holds 16 rows m of one column; its two columns
// are neighbours (n = 2 (lane & 31) + j), so a wave's access to a row of y is 64 contiguous
// elements.  A lane reads its part of y before anything is stored: y_out may be y_in, so reads left
// among the stores waited for memory one after another.
// SPLIT waves share a block, each making its products again and finishing 16 / SPLIT of a lane's rows:
// a small grid is bound by one wave's chain of activations and stores (lora_epilogue_split).
template <typename YI, typename YO, bool DRB, int SPLIT>
__global__ __launch_bounds__(256) void lora_epilogue_kernel(LinearEpilogueArgs a, int64_t tiles_n) {
  constexpr int RPW = 16 / SPLIT;  // rows of a lane that this wave finishes: v0 .. v0 + RPW - 1
  const int lane = threadIdx.x & 63, r32 = lane & 31, half = lane >> 5;
  const int64_t w = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int v0 = (int)(w % SPLIT) * RPW;
  const int64_t m0 = w / SPLIT / tiles_n * 32, n0 = w / SPLIT % tiles_n * 64;
  if (m0 >= a.M) return;  // waves past the last block
  const int64_t mr = m0 + r32 < a.M ? m0 + r32 : a.M - 1;  // rows and columns past the ends repeat
  int64_t nr[2];                                           // the last one and are never stored
#pragma unroll
  for (int j = 0; j < 2; ++j) nr[j] = n0 + 2 * r32 + j < a.N ? n0 + 2 * r32 + j : a.N - 1;
  const int64_t n = n0 + 2 * r32;
  const YI* const yi = static_cast<const YI*>(a.y_in);
  YO* const yo = static_cast<YO*>(a.y_out);
  struct alignas(2 * sizeof(YI)) VI { YI v[2]; };
  struct alignas(2 * sizeof(YO)) VO { YO v[2]; };
  // Pairs need an even N (a row's start aligned to two elements); both pointers are.
  const bool pairs = a.N % 2 == 0 && reinterpret_cast<uintptr_t>(a.y_in) % sizeof(VI) == 0 &&
                     reinterpret_cast<uintptr_t>(a.y_out) % sizeof(VO) == 0;
  auto row = [&](int v) { return m0 + 8 * ((v0 + v) >> 2) + 4 * half + ((v0 + v) & 3); };
  VI in[RPW];
  if (pairs) {
#pragma unroll
    for (int v = 0; v < RPW; ++v)
      in[v] = *reinterpret_cast<const VI*>(yi + (row(v) < a.M ? row(v) : a.M - 1) * a.N + (n < a.N ? n : a.N - 2));
  } else {
#pragma unroll
    for (int v = 0; v < RPW; ++v)
#pragma unroll
      for (int j = 0; j < 2; ++j) in[v].v[j] = yi[(row(v) < a.M ? row(v) : a.M - 1) * a.N + nr[j]];
  }
  f32x16 r[2] = {f32x16{}, f32x16{}};
  for (int k = 0; k < a.R; k += 16) {
    if constexpr (DRB) {
      const bf16x8 xv = *reinterpret_cast<const bf16x8*>(static_cast<const uint16_t*>(a.xa) + mr * a.R + k + 8 * half);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const bf16x8 bv = *reinterpret_cast<const bf16x8*>(static_cast<const uint16_t*>(a.lbt) + nr[j] * a.R + k + 8 * half);
        r[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xv, bv, r[j], 0, 0, 0);
      }
    } else {
      const float* xp = static_cast<const float*>(a.xa) + mr * a.R + k + 8 * half;
      const f32x4 x0 = *reinterpret_cast<const f32x4*>(xp), x1 = *reinterpret_cast<const f32x4*>(xp + 4);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float* bp = static_cast<const float*>(a.lbt) + nr[j] * a.R + k + 8 * half;
        const f32x4 b0 = *reinterpret_cast<const f32x4*>(bp), b1 = *reinterpret_cast<const f32x4*>(bp + 4);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          r[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x0[t], b0[t], r[j], 0, 0, 0);
          r[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x1[t], b1[t], r[j], 0, 0, 0);
        }
      }
    }
  }
  if (n >= a.N) return;
  float rv[2][RPW];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int v = 0; v < RPW; ++v) {
      rv[j][v] = r[j][v];
#pragma unroll
      for (int s = 1; s < SPLIT; ++s) rv[j][v] = v0 == s * RPW ? r[j][s * RPW + v] : rv[j][v];
    }
#pragma unroll
  for (int v = 0; v < RPW; ++v) {
    if (row(v) >= a.M) continue;
    const int64_t t = row(v) * a.N + n;
    if (pairs) {
      VO out;
#pragma unroll
      for (int j = 0; j < 2; ++j) Act<YO>::st(out.v, j, epilogue_finish(a, Act<YI>::ld(in[v].v, j), n + j, true, rv[j][v]));
      *reinterpret_cast<VO*>(yo + t) = out;
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (n + j < a.N) Act<YO>::st(yo, t + j, epilogue_finish(a, Act<YI>::ld(in[v].v, j), n + j, true, rv[j][v]));
    }
  }
}

// Waves per 32 x 64 block.  Same-process times in us for 1 / 4 / 16 (whole calls; one thread per output in
// brackets): 36 blocks, [66, 1024] rank 1 with GELU 20.9 / - / - [16.2]; 16 blocks, [28, 640] rank 8
// 10.7 / 6.9 / 5.7 [8.5]; 64 blocks, [11, 832] rank 16 17.2 / 15.6 / 14.0 [16.7]; 124 blocks, [98, 1216]
// rank 1 with GELU 26.5 / 20.5 / 19.2 [24.5]; 101 blocks, [5, 704] rank 256 30.9 / 29.3 / 40.2; 365 blocks,
// [140, 1792] rank 64 39.1 / 31.0 / 34.5; 560 blocks, [233, 832] rank 256 63.0 / 65.7 / 96.5; 814 blocks, rank
// 256 61.6 / 91.4 / 188.
static int lora_epilogue_split(int64_t tiles) { return tiles <= 64 ? 16 : tiles <= 512 ? 4 : 1; }

int run_linear_epilogue(const LinearEpilogueArgs& a, hipStream_t st) {
  const int64_t total = a.M * a.N;
  if (total == 0) return MLXQ_OK;
  const int64_t blocks = (total + 255) / 256;
  if (blocks > 0x7fffffff) return set_error(MLXQ_EINVAL, "linear epilogue: problem too large");
  const bool table_act = a.act == MLXQ_ACT_GELU_TANH || a.act == MLXQ_ACT_GELU_EXACT;
  if (table_act && a.d2_bf16 && a.act_table == nullptr)
    return set_error(MLXQ_EINVAL, "linear epilogue: activation table missing");
  const dim3 b(256);
  if (a.R > 0) {
    const int64_t tiles_n = (a.N + 63) / 64, tiles = (a.M + 31) / 32 * tiles_n;
    const int split = lora_epilogue_split(tiles);
    const dim3 g((unsigned)((tiles * split + 3) / 4));
#define MLXQ_LES(YI, YO, S)                                                                             \
  do {                                                                                                  \
    if (a.dr_bf16) hipLaunchKernelGGL((lora_epilogue_kernel<YI, YO, true, S>), g, b, 0, st, a, tiles_n); \
    else hipLaunchKernelGGL((lora_epilogue_kernel<YI, YO, false, S>), g, b, 0, st, a, tiles_n);         \
  } while (0)
#define MLXQ_LE(YI, YO)                     \
  do {                                      \
    if (split == 1) MLXQ_LES(YI, YO, 1);    \
    else if (split == 4) MLXQ_LES(YI, YO, 4); \
    else MLXQ_LES(YI, YO, 16);              \
  } while (0)
    if (a.y_in_bf16 && a.y_out_bf16) MLXQ_LE(uint16_t, uint16_t);
    else if (a.y_in_bf16) MLXQ_LE(uint16_t, float);
    else if (a.y_out_bf16) MLXQ_LE(float, uint16_t);
    else MLXQ_LE(float, float);
#undef MLXQ_LE
#undef MLXQ_LES
    return check_launch("linear_epilogue");
  }
  const dim3 g((unsigned)blocks);
  if (a.y_in_bf16 && a.y_out_bf16) hipLaunchKernelGGL((linear_epilogue_kernel<uint16_t, uint16_t>), g, b, 0, st, a);
  else if (a.y_in_bf16) hipLaunchKernelGGL((linear_epilogue_kernel<uint16_t, float>), g, b, 0, st, a);
  else if (a.y_out_bf16) hipLaunchKernelGGL((linear_epilogue_kernel<float, uint16_t>), g, b, 0, st, a);
  else hipLaunchKernelGGL((linear_epilogue_kernel<float, float>), g, b, 0, st, a);
  return check_launch("linear_epilogue");
}

// dst[i] = src[i] converted between f32 and bf16 (round to nearest even) or copied.
template <typename ST, typename DT>
__global__ void cast_kernel(const ST* __restrict__ src, DT* __restrict__ dst, int64_t n) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) Act<DT>::st(dst, t, Act<ST>::ld(src, t));
}

int run_cast(const void* src, int src_dtype, void* dst, int dst_dtype, int64_t n, hipStream_t st) {
  if (n == 0) return MLXQ_OK;
  const int64_t blocks = (n + 255) / 256;
  if (blocks > 0x7fffffff) return set_error(MLXQ_EINVAL, "cast: %lld elements is too many", (long long)n);
  const dim3 g((unsigned)blocks), b(256);
  if (src_dtype == MLXQ_BFLOAT16 && dst_dtype == MLXQ_BFLOAT16)
    hipLaunchKernelGGL((cast_kernel<uint16_t, uint16_t>), g, b, 0, st, (const uint16_t*)src, (uint16_t*)dst, n);
  else if (src_dtype == MLXQ_BFLOAT16)
    hipLaunchKernelGGL((cast_kernel<uint16_t, float>), g, b, 0, st, (const uint16_t*)src, (float*)dst, n);
  else if (dst_dtype == MLXQ_BFLOAT16)
    hipLaunchKernelGGL((cast_kernel<float, uint16_t>), g, b, 0, st, (const float*)src, (uint16_t*)dst, n);
  else
    hipLaunchKernelGGL((cast_kernel<float, float>), g, b, 0, st, (const float*)src, (float*)dst, n);
  return check_launch("cast");
}

}  // namespace mlxq
