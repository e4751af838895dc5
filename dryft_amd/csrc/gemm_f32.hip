// Matrix products of the float32 path, y[M,N] = x[M,K] . W[N,K]^T, on the matrix cores' full-precision instruction
// (v_mfma_f32_16x16x4_f32: 32-bit factors, 32-bit sums). A lane's 16 bytes of a row are four values of K, one for each of
// four instructions; which values of K meet in one instruction does not matter to the sum, so lane (c, g) takes piece g of
// every four pieces of its row, for both operands alike.
//
//  * gemm_few_f32: at most 16 rows of x (decoding). Bound by reading W once.
//  * gemm_direct_f32: any number of rows. Bound by the instruction: 256 flops a clock and compute unit.
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ f32x4 mfma4(f32x4 a, f32x4 b, f32x4 acc) {
#pragma unroll
  for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], acc, 0, 0, 0);
  return acc;
}

// ------------------------------------------------------------------------------------------- few rows
// A workgroup takes 16 rows of W and its WAVES waves split K in runs of whole blocks of 32 values (a 128-byte line of a
// row), four blocks of both operands in flight; the waves' sums meet in LDS and are added in the order 0, 1, .... With GLU
// the 16 rows are the gate rows of eight outputs and their up rows, and y = silu(gate) * up.
// The step's matrices are small (4 to 25 MB), so what counts is how many trips to memory a wave makes one after the other:
// Qwen3-0.6B's at 4 rows in a captured step, us, against the plain kernel
// below (two rows of W a wave, each wave walking all of K with a barrier every 256 values), which served all of them before:
// q/k/v 6.6 (8.1), o in four runs of K 4.6 (10.1), gate/up with its activation 9.9 (9.4 and 4.7 for the activation), down in
// four runs 6.4 (13.7).
#define FEW_BLOCKS 4
// Products of few outputs also split K over gridDim.y workgroups: y is then [gridDim.y, M, N], sums that the consumer adds.
template <int WAVES, bool GLU>
__global__ __launch_bounds__(WAVES * WAVE) void gemm_few_f32_kernel(const float* __restrict__ x, int64_t x_stride,
                                                                    const float* __restrict__ w, float* __restrict__ y,
                                                                    int M, int N, int K) {
  __shared__ f32x4 sums[WAVES][WAVE];
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE, c = lane % 16, g = lane / 16;
  constexpr int OUTS = GLU ? 8 : 16;
  const int n0 = blockIdx.x * OUTS;
  const int64_t w_row = GLU ? (c < 8 ? 0 : N) + min(n0 + (c & 7), N - 1) : min(n0 + c, N - 1);
  const float* wp = w + w_row * K;
  const float* xp = x + (int64_t)min(c, M - 1) * x_stride;
  const int units = WAVES * gridDim.y, per = ((K + 31) / 32 + units - 1) / units * 32;
  const int k_begin = min((int)(blockIdx.y * WAVES + wave) * per, K), k_end = min(k_begin + per, K);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = k_begin; k0 < k_end; k0 += 32 * FEW_BLOCKS) {
    f32x4 wv[2 * FEW_BLOCKS], xv[2 * FEW_BLOCKS];
#pragma unroll
    for (int u = 0; u < 2 * FEW_BLOCKS; ++u) {
      const int k = k0 + 16 * u + 4 * g, kk = min(k, K - 4);       // K is a multiple of 4; beyond the run: times zeros
      wv[u] = *(const f32x4*)(wp + kk);
      xv[u] = *(const f32x4*)(xp + kk);
      if (k >= k_end) xv[u] = zero, wv[u] = zero;
    }
    __builtin_amdgcn_sched_barrier(0);                             // every load of the four blocks before the first product
#pragma unroll
    for (int u = 0; u < 2 * FEW_BLOCKS; ++u) acc = mfma4(wv[u], xv[u], acc);
  }
  sums[wave][lane] = acc;
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int v = 1; v < WAVES; ++v) acc += sums[v][lane];
  // acc[i] is row 4g + i of the workgroup's 16 for row c of x
  if (GLU) {
    f32x4 up;
#pragma unroll
    for (int i = 0; i < 4; ++i) up[i] = __shfl_xor(acc[i], 32, WAVE);
    if (g >= 2 || c >= M) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = n0 + 4 * g + i;
      if (n < N) y[(int64_t)c * N + n] = acc[i] / (1.f + expf(-acc[i])) * up[i];
    }
    return;
  }
  if (c >= M) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int n = n0 + 4 * g + i;
    if (n < N) y[((int64_t)blockIdx.y * M + c) * N + n] = acc[i];
  }
}

template <bool GLU>
static int launch_few(const float* x, int64_t x_stride, const float* w, float* y, int M, int N, int K, int splits,
                      hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 16 || K <= 0 || K % 4 || x_stride % 4 || (((uintptr_t)x | (uintptr_t)w) & 15) || splits < 1 || splits > 64) return -1;
  const int outs = GLU ? 8 : 16;
  const dim3 grid((N + outs - 1) / outs, splits);
#define FEW(W) hipLaunchKernelGGL((gemm_few_f32_kernel<W, GLU>), grid, dim3(W * WAVE), 0, stream, x, x_stride, w, y, M, N, K)
  // a wave takes four blocks of K or so; few workgroups walk a long K in twice as many waves
  if (K <= 512 * splits) FEW(4);
  else if (grid.x * splits < 256 && K >= 2048 * splits) FEW(16);
  else FEW(8);
#undef FEW
  return DRYFT_LAUNCH_CHECK();
}

// M <= 16, K and x_stride multiples of 4, x and W at 16-byte addresses. splits > 1: y is [splits, M, N], sums over as many
// runs of K
DRYFT_API int dryft_gemm_rows_f32(const void* x, int64_t x_stride, const void* w, void* y, int M, int N, int K, int splits,
                                  hipStream_t stream) {
  return launch_few<false>((const float*)x, x_stride, (const float*)w, (float*)y, M, N, K, splits, stream);
}

// y[M, N] = silu(x . Wg^T) * (x . Wu^T) with W = [Wg; Wu] of 2N rows; the rest as above
DRYFT_API int dryft_gemm_rows_swiglu_f32(const void* x, int64_t x_stride, const void* w, void* y, int M, int N, int K,
                                         hipStream_t stream) {
  return launch_few<true>((const float*)x, x_stride, (const float*)w, (float*)y, M, N, K, 1, stream);
}

// ------------------------------------------------------------------------------------------- few rows, many outputs
// At most 16 rows again, where there are workgroups enough: plain multiply-adds. A workgroup owns 8 weight rows, two per
// wave, and walks K in chunks of 256: the rows of x for a chunk are staged in LDS once for all four waves (double-buffered,
// one barrier per chunk), a lane takes four consecutive values of each of its weight rows (16-byte loads, a wave reads 1 KB of
// a row per instruction; the next chunk's are in flight while this one is multiplied) and the matching four of every row of
// x. At the end the 64 lanes' sums are added. K must be a multiple of 4; rows beyond N are read from a clamped row, never
// stored. Bound by memory at up to four rows (the output head of
// Qwen3-0.6B, 622 MB: 105 us at one row, 5.9 TB/s), by the multiply-adds beyond (352 us at 16 rows).
#define ROWS_CHUNK 256
template <int MR>
__global__ __launch_bounds__(256) void gemm_stream_f32_kernel(const float* __restrict__ x, int64_t x_stride,
                                                            const float* __restrict__ w, float* __restrict__ y, int M,
                                                            int N, int K) {
  __shared__ __align__(16) float xs[2][MR][ROWS_CHUNK + 4];
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
  const int n0 = blockIdx.x * 8 + 2 * wave;
  const float* w_row[2] = {w + (int64_t)min(n0, N - 1) * K, w + (int64_t)min(n0 + 1, N - 1) * K};
  float acc[2][MR];
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int m = 0; m < MR; ++m) acc[r][m] = 0.f;
  float xr[MR];                                            // thread t brings value k0 + t of every row of x
  auto fetch_x = [&](int k0) {                             // beyond K or M: a valid address, stored as zero
    const int k = min(k0 + (int)threadIdx.x, K - 1);
#pragma unroll
    for (int m = 0; m < MR; ++m) xr[m] = x[(int64_t)min(m, M - 1) * x_stride + k];
  };
  auto store_x = [&](int buf, int k0) {
    const bool in = k0 + (int)threadIdx.x < K;
#pragma unroll
    for (int m = 0; m < MR; ++m) xs[buf][m][threadIdx.x] = (in && m < M) ? xr[m] : 0.f;
  };
  f32x4 wv[2], wn[2];
  auto fetch = [&](f32x4 (&v)[2], int k0) {                // beyond K: the row's last four values, multiplied by zeros
    const int kk = min(k0 + 4 * lane, K - 4);
    v[0] = *(const f32x4*)(w_row[0] + kk);
    v[1] = *(const f32x4*)(w_row[1] + kk);
  };
  fetch_x(0);
  fetch(wv, 0);
  store_x(0, 0);
  int buf = 0;
  for (int k0 = 0; k0 < K; k0 += ROWS_CHUNK, buf ^= 1) {
    __syncthreads();                                       // the chunk is staged; the other buffer is free again
    fetch_x(k0 + ROWS_CHUNK);                              // the next chunk's loads are in flight during the products
    fetch(wn, k0 + ROWS_CHUNK);
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const f32x4 xv = *(const f32x4*)&xs[buf][m][4 * lane];   // zeros beyond K
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[r][m] = fmaf(wv[r][i], xv[i], acc[r][m]);
    }
    store_x(buf ^ 1, k0 + ROWS_CHUNK);
    wv[0] = wn[0];
    wv[1] = wn[1];
  }
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const float s = wave_sum(acc[r][m]);
      if (lane == 0 && m < M && n0 + r < N) y[(int64_t)m * N + n0 + r] = s;
    }
}

// M <= 16, K a multiple of 4, W at a 16-byte address
DRYFT_API int dryft_gemm_stream_f32(const void* x, int64_t x_stride, const void* w, void* y, int M, int N, int K,
                                    hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 16 || K <= 0 || K % 4 || ((uintptr_t)w & 15)) return -1;
  dim3 grid((N + 7) / 8), block(256);
#define RW(MRV)                                                                                                \
  hipLaunchKernelGGL(gemm_stream_f32_kernel<MRV>, grid, block, 0, stream, (const float*)x, x_stride, (const float*)w, \
                     (float*)y, M, N, K)
  if (M <= 1) RW(1);
  else if (M <= 2) RW(2);
  else if (M <= 4) RW(4);
  else if (M <= 8) RW(8);
  else RW(16);
#undef RW
  return DRYFT_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------------------------- any number of rows
// Four waves own a block of 32 MT rows of x by 32 NT rows of W, a wave MT x NT tiles of 16 x 16. K goes by in steps of 32
// values: 128 bytes of every row, brought straight into LDS (global_load_lds_dwordx4), STAGES - 1 steps ahead of the one
// that is multiplied, piece p of row r at place p ^ ((r / 2) % 8) so that operand reads meet no bank twice. Every wave
// issues the same number of loads per step, also past the end of K (the last step again, into a buffer nobody reads), so
// one constant says how many may be in flight.
// The block's size is what the launcher chooses by the number of workgroups (dryft_gemm_direct_f32_shape): the instruction is
// the bound, 32 x 32 outputs a wave read LDS less than a quarter of the time, so a smaller block costs nothing but trips to
// the caches and divides the work evenly where large ones leave compute units idle. Qwen3-0.6B's products at 525 rows in a
// captured step, us, blocks of 128 x 128 / 64 x 64 / 32 x 64, and before, 128 x 128 through registers: q/k/v 69 / 54 / 47 (82),
// o 133 / 40 / 38 (156), gate/up 70 / 71 / 64 (83), down 197 / 60 / 55 (227), output head 1,608 / 1,611 / 2,180 (1,648);
// at 32 rows q/k/v 67 / 22 / 14 (77), down 193 / 58 / 35 (219). The best of each is 58 to 117 of the 157 TFLOP/s.
#define DIRECT_STEP_BYTES 128

__device__ __forceinline__ void load16_to_lds(const void* base, uint32_t offset, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_base), "v"(offset), "s"(base) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void wait_loads() {             // all but the last N have arrived
  __builtin_amdgcn_s_waitcnt(0x0f70 | (N & 15) | ((N >> 4) << 14));
  asm volatile("" ::: "memory");
}

template <int MT, int NT, int STAGES>
__global__ __launch_bounds__(256) void gemm_direct_f32_kernel(const float* __restrict__ x, int64_t x_stride,
                                                              const float* __restrict__ w, float* __restrict__ y, int M,
                                                              int N, int K) {
  extern __shared__ __align__(16) unsigned char direct_lds[];
  constexpr int RB = DIRECT_STEP_BYTES, BM = 32 * MT, BN = 32 * NT;
  constexpr int X_BYTES = BM * RB, STAGE_BYTES = (BM + BN) * RB;
  constexpr int X_LOADS = MT, W_LOADS = NT, LOADS = X_LOADS + W_LOADS;     // of 1 KB (8 rows) per wave and step
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE, c = lane % 16, g = lane / 16;
  const int wm = wave / 2, wn = wave % 2;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN, steps = K / 32;
  uint32_t x_from[X_LOADS], w_from[W_LOADS];
#pragma unroll
  for (int i = 0; i < X_LOADS; ++i) {
    const int r = 8 * (wave + 4 * i) + lane / 8;           // row of the block's part of x
    x_from[i] = (uint32_t)min(m0 + r, M - 1) * (uint32_t)x_stride * 4u + (((lane % 8) ^ ((r >> 1) & 7)) << 4);
  }
#pragma unroll
  for (int i = 0; i < W_LOADS; ++i) {
    const int r = 8 * (wave + 4 * i) + lane / 8;
    w_from[i] = (uint32_t)min(n0 + r, N - 1) * (uint32_t)K * 4u + (((lane % 8) ^ ((r >> 1) & 7)) << 4);
  }
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)direct_lds);
  auto fetch = [&](int step, int stage) {
    const int64_t at = (int64_t)min(step, steps - 1) * RB;
    const uint32_t to = lds0 + stage * STAGE_BYTES;
#pragma unroll
    for (int i = 0; i < X_LOADS; ++i) load16_to_lds((const unsigned char*)x + at, x_from[i], to + (wave + 4 * i) * 1024);
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) load16_to_lds((const unsigned char*)w + at, w_from[i], to + X_BYTES + (wave + 4 * i) * 1024);
  };
  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s) fetch(s, s);
  int stage = 0;
  const int sw = (c >> 1) & 7;                             // row 16 t + c of any tile is swizzled like row c
  for (int step = 0; step < steps; ++step) {
    wait_loads<(STAGES - 2) * LOADS>();                    // this step has arrived
    __syncthreads();                                       // everybody's part of it too; the step before is done with
    fetch(step + STAGES - 1, stage == 0 ? STAGES - 1 : stage - 1);
    const unsigned char* xs = direct_lds + stage * STAGE_BYTES + (16 * MT * wm + c) * RB;
    const unsigned char* ws = direct_lds + stage * STAGE_BYTES + X_BYTES + (16 * NT * wn + c) * RB;
#pragma unroll
    for (int u = 0; u < 2; ++u) {                          // 16 values of K at a time
      const int place = ((4 * u + g) ^ sw) << 4;
      f32x4 a[NT], b[MT];
#pragma unroll
      for (int t = 0; t < NT; ++t) a[t] = *(const f32x4*)(ws + 16 * t * RB + place);
#pragma unroll
      for (int t = 0; t < MT; ++t) b[t] = *(const f32x4*)(xs + 16 * t * RB + place);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
            acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[nt][i], b[mt][i], acc[mt][nt], 0, 0, 0);
    }
    stage = stage + 1 == STAGES ? 0 : stage + 1;
  }
  wait_loads<0>();                                         // the loads past the end have landed before the waves leave
  // acc[mt][nt][i] is output (tile nt) + 4g + i of row (tile mt) + c
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = m0 + 16 * (MT * wm + mt) + c;
    if (m >= M) continue;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int n = n0 + 16 * (NT * wn + nt) + 4 * g;
      if (n + 3 < N && (N & 3) == 0) {
        *(f32x4*)(y + (int64_t)m * N + n) = acc[mt][nt];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < N) y[(int64_t)m * N + n + i] = acc[mt][nt][i];
      }
    }
  }
}

template <int MT, int NT, int STAGES>
static int launch_direct(const float* x, int64_t x_stride, const float* w, float* y, int M, int N, int K, hipStream_t stream) {
  constexpr int BM = 32 * MT, BN = 32 * NT, lds = STAGES * (BM + BN) * DIRECT_STEP_BYTES;
  static_assert(lds <= 160 * 1024, "the stages must fit a compute unit's LDS");
  auto kernel = gemm_direct_f32_kernel<MT, NT, STAGES>;
  static bool raised = false;                              // more dynamic LDS than the default limit allows
  if (lds > 64 * 1024 && !raised) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return -2;
    raised = true;
  }
  dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM);
  if (grid.y > 65535) return -1;
  hipLaunchKernelGGL(kernel, grid, dim3(256), lds, stream, x, x_stride, w, y, M, N, K);
  return DRYFT_LAUNCH_CHECK();
}

// Which block: 0 = 128 x 128, 1 = 64 x 64, 2 = 32 x 64 (rows of x by rows of W): the one whose busiest compute unit has the
// fewest outputs to do, the larger one where two are within a twelfth (it reads the caches less). Blocks of few rows do not
// take more rows than a grid has places for them.
DRYFT_API int dryft_gemm_direct_f32_shape(int M, int N) {
  const int bm[3] = {128, 64, 32}, bn[3] = {128, 64, 64};
  int best = 0;
  double least = 1e30;
  for (int s = 0; s < 3; ++s) {
    if (((int64_t)M + bm[s] - 1) / bm[s] > 65535) continue;
    const int64_t blocks = (int64_t)((M + bm[s] - 1) / bm[s]) * ((N + bn[s] - 1) / bn[s]);
    const double work = (double)((blocks + 255) / 256) * bm[s] * bn[s];
    if (work < least * (11.0 / 12.0)) {
      least = work;
      best = s;
    }
  }
  return best;
}

// K a multiple of 32, x_stride of 4, operands at 16-byte addresses and within 4 GiB from their start. shape -1: chosen here
DRYFT_API int dryft_gemm_direct_f32(const void* x, int64_t x_stride, const void* w, void* y, int M, int N, int K, int shape,
                                    hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || K % 32 || x_stride % 4 || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) ||
      (int64_t)N * K * 4 >= (int64_t)4 << 30 || (int64_t)M * x_stride * 4 >= (int64_t)4 << 30)
    return -1;
  const float *xf = (const float*)x, *wf = (const float*)w;
  switch (shape < 0 ? dryft_gemm_direct_f32_shape(M, N) : shape) {
    case 0: return launch_direct<4, 4, 3>(xf, x_stride, wf, (float*)y, M, N, K, stream);
    case 1: return launch_direct<2, 2, 4>(xf, x_stride, wf, (float*)y, M, N, K, stream);
    case 2: return launch_direct<1, 2, 4>(xf, x_stride, wf, (float*)y, M, N, K, stream);
    default: return -1;
  }
}
