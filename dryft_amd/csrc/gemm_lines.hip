// Matrix products of at most 16 rows in bfloat16, 4 in float32, whose sums are whole when a workgroup ends: y[M,N] = x[M,K] . W[N,K]^T, and the
// gated units of feed-forwards on top of such products.
//
// Decoding steps are chains of launches, each too short to hide the trips to memory at its ends, so this kernel is built to
// make as few of them as it can and to leave nothing for a launch of its own afterwards:
//
//  * A load instruction brings four weight rows, 256 contiguous bytes of each, and its registers are a matrix-core operand
//    as they are. v_mfma_f32_16x16x32_bf16 takes 16 rows of 32 values; "row" c of the operand is here piece c % 4 of weight
//    row c / 4 (8 values of every 32), and the rows of x are cut the same way. Of the 16 x 16 products those of equal pieces
//    count: a quarter of the matrix cores' work, of which there is plenty, buys whole cache lines without a way through LDS.
//    (Eight pieces of two rows: 1 to 3 % faster at one row, 5 to 15 % slower at four and eight.)
//  * K is split over the waves of a workgroup (blocks of 128 values in turn, so that together they read on without gaps) and
//    over nothing else; the waves' sums meet in LDS.
//  * The end of the kernel may be what a layer does next: the residual sum r <- T(r + y) and each workgroup's sums of r^2
//    (`Residual`). The next product, given r and those sums (`LateNorm`), takes its rows through the norm on their way to the matrix
//    cores, T(T(r * rsqrt(mean(r^2) + eps)) * weight) as the norm's own kernel rounds, while its weights are on their way: the norm
//    between two products needs no launch.
//
// Bound by the weights' bytes and by the two ends of a launch. In a captured chain on rotating cold weights, us at 1 / 4 / 8 rows,
// against the line-staging kernel with its splits of K: 2,560 x 4,096 5.7 / 5.8 / 6.2 (6.4 / 6.3 / 6.6), 2,560 x 9,728 10.1 / 10.3 /
// 10.9 (11.4 / 11.5 / 11.8), 6,144 x 2,560 7.3 / 7.3 / 8.0 (8.1 / 8.2 / 8.5), 1,024 x 3,072 3.7 / 3.8 / 4.3 (4.2 / 4.3 / 4.4), 2,048 x
// 2,048 4.0 / 4.0 / 4.1 (4.5), 8,192 x 2,048 7.5 / 7.5 / 8.5 (9.2 / 9.3 / 9.4), 2,048 x 8,192 8.1 / 8.3 / 8.5 (8.7 / 8.8 / 9.0), 65,536 x
// 2,048 42 / 42 / 45 (51 / 50 / 51), 151,936 x 2,560 115 / 121 / 132 (126 / 134 / 147).
// The norm on the way, instead of launches of its own (3.4 to 4.6 us and the gap before each, two a layer), whole passes of 96
// decoding steps through 12 layers of Qwen3-4B: one sequence 79.7 -> 73.5 ms, eight 135.4 -> 131.2 ms; 64 steps of three sequences
// through Qwen3-0.6B 62.6 -> 56.4 ms.
#include "gate_unit.h"
#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

#define LINES_ROWS 16          // the most rows of x, in bfloat16
#define LINES_ROWS_F32 4       // and in float32
#define LATE_ROWS 8            // rows that the sums of squares have places for: squares[count][LATE_ROWS]
#define LATE_MOST 1024         // workgroups that may have left sums

template <typename E>
struct LateNorm {
  const float* squares = nullptr;
  int count = 0;
  float eps = 0.f;
  const E* weight = nullptr;
};

template <typename E>
struct Residual {
  E* rows = nullptr;                // r, updated in place; null: the product is stored
  float* squares = nullptr;
};

// Further products of the same rows in the same launch, workgroups of their own behind the first product's: small ones (gates, step
// sizes, low-rank projections) are all trips to memory as launches of their own.
#define LINES_BESIDE 3
template <typename E>
struct Beside {
  int count = 0;
  const E* w[LINES_BESIDE] = {};
  void* y[LINES_BESIDE] = {};
  int n[LINES_BESIDE] = {}, y_f32[LINES_BESIDE] = {};
};

// Sixteen bytes of a row are an operand of one matrix instruction of 32 values in bfloat16, or a value for each of four
// instructions of four values in float32 (32-bit factors and sums).
template <typename E>
struct Fragment;
template <>
struct Fragment<bf16_t> {
  typedef bf16x8 type;
  static constexpr int VALUES = 8;
  static constexpr int SUMS = 1;
  static __device__ __forceinline__ void multiply(bf16x8 a, bf16x8 b, f32x4 (&acc)[SUMS]) {
    acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[0], 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 sum(const f32x4 (&acc)[SUMS]) { return acc[0]; }
  static __device__ __forceinline__ bf16x8 zero() {
    bf16x8 z;
#pragma unroll
    for (int i = 0; i < 8; ++i) z[i] = (__bf16)0.f;
    return z;
  }
  // a fragment of a row through the norm: T(T(r * inverse) * weight)
  static __device__ __forceinline__ bf16x8 normed(bf16x8 r, float inverse, bf16x8 weight) {
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = (__bf16)((float)(__bf16)((float)r[i] * inverse) * (float)weight[i]);
    return r;
  }
};
template <>
struct Fragment<float> {
  typedef f32x4 type;
  static constexpr int VALUES = 4;
  // a sum for each of the four: no instruction waits for the one before, and sums a quarter as long are rounded less (against 64
  // bits, relative to the result's norm, K = 1,024: 1.0e-7 instead of 1.6e-7; 9,728: 1.8e-7 instead of 3.3e-7)
  static constexpr int SUMS = 4;
  static __device__ __forceinline__ void multiply(f32x4 a, f32x4 b, f32x4 (&acc)[SUMS]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], acc[i], 0, 0, 0);
  }
  static __device__ __forceinline__ f32x4 sum(const f32x4 (&acc)[SUMS]) { return (acc[0] + acc[1]) + (acc[2] + acc[3]); }
  static __device__ __forceinline__ f32x4 zero() { return f32x4{0.f, 0.f, 0.f, 0.f}; }
  static __device__ __forceinline__ f32x4 normed(f32x4 r, float inverse, f32x4 weight) {
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = r[i] * inverse * weight[i];
    return r;
  }
};

template <int N, int I = 0, typename F>
__device__ __forceinline__ void each(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    each<N, I + 1>(f);
  }
}

// ROWS weight rows a workgroup (with GLU half of them gate rows and then their up rows), X groups of four rows of x, DEPTH blocks
// of 256 bytes of K of a wave on their way at a time
template <typename E, int ROWS, int X, int WAVES, int DEPTH, bool GLU, bool LATE, bool MORE>
__global__ __launch_bounds__(64 * WAVES) void gemm_lines_kernel(const E* __restrict__ x, int64_t x_stride,
                                                                const E* __restrict__ w, void* __restrict__ y, int y_f32,
                                                                int M, int N, int K, LateNorm<E> late, Residual<E> residual,
                                                                GateAct act, Beside<E> beside) {
  typedef Fragment<E> F;
  typedef typename F::type frag;
  constexpr int T = (ROWS + 3) / 4, BLOCK = 16 * F::VALUES, OUT = GLU ? ROWS / 2 : ROWS;
  __shared__ float sums[WAVES][T][X][4][4], late_sums[LATE ? WAVES : 1][LATE_ROWS], squares[GLU ? 1 : ROWS][LATE_ROWS];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
  const int c = lane % 16, g = lane / 16, piece = c % 4;
  int block = blockIdx.x;
  if constexpr (MORE) {                                    // whose outputs these are
#pragma unroll
    for (int p = 0; p < LINES_BESIDE; ++p) {
      const int blocks = (N + OUT - 1) / OUT;
      if (p < beside.count && block >= blocks) {
        block -= blocks;
        w = beside.w[p];
        y = beside.y[p];
        N = beside.n[p];
        y_f32 = beside.y_f32[p];
      }
    }
  }
  const int n0 = block * OUT;
  f32x4 late_held[X];                                      // sums of squares, asked for ahead of everything
  if constexpr (LATE) {
#pragma unroll
    for (int i = 0; i < X; ++i) {
      late_held[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int from = threadIdx.x + 64 * WAVES; from < late.count; from += 64 * WAVES)
        late_held[i] += *(const f32x4*)(late.squares + from * LATE_ROWS + 4 * i);
    }
    const int from = min((int)threadIdx.x, late.count - 1);
#pragma unroll
    for (int i = 0; i < X; ++i) {
      const f32x4 one = *(const f32x4*)(late.squares + from * LATE_ROWS + 4 * i);
#pragma unroll
      for (int j = 0; j < 4; ++j) late_held[i][j] += (int)threadIdx.x < late.count ? one[j] : 0.f;
    }
  }
  const int at = F::VALUES * (4 * g + piece);                       // of this lane within a block
  const E* wp[T];
  const E* xp[X];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int row = min(4 * t + c / 4, ROWS - 1);          // past the workgroup's rows and the matrix's: the last one again
    wp[t] = w + (int64_t)(GLU && row >= OUT ? N + min(n0 + row - OUT, N - 1) : min(n0 + row, N - 1)) * K;
  }
#pragma unroll
  for (int i = 0; i < X; ++i) xp[i] = x + (int64_t)min(4 * i + c / 4, M - 1) * x_stride;
  f32x4 acc[T][X][F::SUMS];
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int i = 0; i < X; ++i)
#pragma unroll
      for (int u = 0; u < F::SUMS; ++u) acc[t][i][u] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int blocks = (K + BLOCK - 1) / BLOCK, mine = (blocks - wave + WAVES - 1) / WAVES;    // wave, wave + WAVES, ...
  frag a[DEPTH][T], b[DEPTH][X], norm[LATE ? DEPTH : 1];
  float inverse[X];
  auto fetch = [&](auto slot, int i) {
    constexpr int d = decltype(slot)::value;
    int k = (wave + i * WAVES) * BLOCK + at;
    k = k < K ? k : 0;                                     // beyond K (a multiple of a fragment): any values, zeros when they are used
#pragma unroll
    for (int j = 0; j < X; ++j) b[d][j] = *(const frag*)(xp[j] + k);
    if constexpr (LATE) norm[d] = *(const frag*)(late.weight + k);
#pragma unroll
    for (int t = 0; t < T; ++t) a[d][t] = __builtin_nontemporal_load((const frag*)(wp[t] + k));
  };
  auto multiply = [&](auto slot, int i) {
    constexpr int d = decltype(slot)::value;
    const int k0 = (wave + i * WAVES) * BLOCK;
    if constexpr (LATE) {
#pragma unroll
      for (int j = 0; j < X; ++j) b[d][j] = F::normed(b[d][j], inverse[j], norm[d]);
    }
    if (k0 + BLOCK > K && k0 + at >= K) {
#pragma unroll
      for (int j = 0; j < X; ++j) b[d][j] = F::zero();
#pragma unroll
      for (int t = 0; t < T; ++t) a[d][t] = F::zero();
    }
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int j = 0; j < X; ++j) F::multiply(a[d][t], b[d][j], acc[t][j]);
  };
  // ahead of a norm every slot is filled, past the wave's blocks too (with any values): the compiler then knows how many loads lie
  // behind the sums of squares, and waits for no operand to add those up
  each<DEPTH>([&](auto d) { if (LATE || d.value < mine) fetch(d, d.value); });
  if constexpr (LATE) {
#pragma unroll
    for (int i = 0; i < X; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float v = lanes_sum<16>(late_held[i][j]);
        v += __shfl_xor(v, 16, WAVE);
        v += __shfl_xor(v, 32, WAVE);
        if (lane == 0) late_sums[wave][4 * i + j] = v;
      }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < X; ++i) {
      float v = 0.f;
#pragma unroll
      for (int u = 0; u < WAVES; ++u) v += late_sums[u][4 * i + c / 4];
      inverse[i] = rsqrtf(v / (float)K + late.eps);
    }
  }
  int i = 0;
  for (; i + 2 * DEPTH <= mine; i += DEPTH)
    each<DEPTH>([&](auto d) {
      multiply(d, i + d.value);
      fetch(d, i + d.value + DEPTH);
    });
  for (; i < mine; i += DEPTH)
    each<DEPTH>([&](auto d) {
      if (i + d.value < mine) {
        multiply(d, i + d.value);
        if (i + d.value + DEPTH < mine) fetch(d, i + d.value + DEPTH);
      }
    });
  // a lane holds the products of x's row c / 4, piece c % 4, with the four pieces of weight row g: one of them counts, and the
  // pieces add up over four lanes
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int j = 0; j < X; ++j) {
      const f32x4 s = F::sum(acc[t][j]);
      const float low = (piece & 1) ? s[1] : s[0], high = (piece & 1) ? s[3] : s[2];
      const float one = lanes_sum<4>((piece & 2) ? high : low);
      if (piece == 0) sums[wave][t][j][g][c / 4] = one;
    }
  __syncthreads();
  for (int e = threadIdx.x; e < OUT * 4 * X; e += 64 * WAVES) {
    const int out = e % OUT, m = e / OUT, n = n0 + out;
    float r2 = 0.f;
    if (m < M && n < N) {
      auto whole = [&](int row) {
        float v = 0.f;
#pragma unroll
        for (int u = 0; u < WAVES; ++u) v += sums[u][row / 4][m / 4][row % 4][m % 4];
        return v;
      };
      const float v = whole(out);
      const int64_t place = (int64_t)m * N + n;
      if constexpr (GLU) {
        if constexpr (sizeof(E) == 4) ((float*)y)[place] = v / (1.f + expf(-v)) * whole(out + OUT);
        else ((bf16_t*)y)[place] = gate_unit(v, whole(out + OUT), act);
      } else if (residual.rows != nullptr) {
        const float r = rounded_as<E>(load_as_float(residual.rows + place) + v);
        store_from_float(residual.rows + place, r);
        r2 = r * r;
      } else if (y_f32) {
        ((float*)y)[place] = v;
      } else {
        store_from_float((E*)y + place, v);
      }
    }
    if constexpr (!GLU && X <= 2) squares[out][m] = r2;
  }
  if constexpr (!GLU && X <= 2) {
    if (residual.rows == nullptr) return;
    __syncthreads();
    if (threadIdx.x < 4 * X) {
      float s = 0.f;
#pragma unroll
      for (int u = 0; u < ROWS; ++u) s += squares[u][threadIdx.x];
      residual.squares[(int64_t)blockIdx.x * LATE_ROWS + threadIdx.x] = s;
    }
  }
}

template <typename E, int ROWS, int X, int WAVES, bool GLU, bool LATE, bool MORE = false>
static int launch_lines(const void* x, int64_t x_stride, const void* w, void* y, int y_f32, int M, int N, int K, LateNorm<E> late,
                        Residual<E> residual, GateAct act, hipStream_t stream, const Beside<E>& beside) {
  constexpr int T = (ROWS + 3) / 4, OUT = GLU ? ROWS / 2 : ROWS;
  // registers for the operands on their way: eight waves have 256 a lane, four are to share a compute unit with others
  constexpr int held = 4 * T * X * Fragment<E>::SUMS;
  constexpr int room = (WAVES == 8 || held > 64 ? 232 : held > 32 || LATE ? 164 : 124) - 28 - held - 2 * (T + X) - (LATE ? 5 * X : 0);
  constexpr int fit = room / (4 * (T + X + (LATE ? 1 : 0)));
  constexpr int most = LATE ? 4 : 10, DEPTH = fit < 1 ? 1 : fit > most ? most : fit;
  // Ahead of a norm five to eight rows are work for the vector units too, and waves side by side hide it better than blocks on their
  // way: one block a wave, us at 8 rows against two or three, 6,144 x 2,560 8.4 (10.0), 4,096 x 1,024 5.0 (6.1), 3,072 gated outputs
  // of 1,024 5.5 (6.1); gated outputs of a long K want two (9,728 of 2,560 20.6, with one 21.5).
  int blocks = (N + OUT - 1) / OUT;
  for (int p = 0; p < beside.count; ++p) blocks += (beside.n[p] + OUT - 1) / OUT;
#define GO(D)                                                                                                                  \
  hipLaunchKernelGGL((gemm_lines_kernel<E, ROWS, X, WAVES, D, GLU, LATE, MORE>), dim3(blocks), dim3(64 * WAVES), 0, stream,          \
                     (const E*)x, x_stride, (const E*)w, y, y_f32, M, N, K, late, residual, act, beside)
  if constexpr (LATE && X == 2 && WAVES == 4) {
    if constexpr (GLU) {
      if (K > 1024) {
        GO(DEPTH);
        return DRYFT_LAUNCH_CHECK();
      }
    }
    GO(1);
  } else {
    GO(DEPTH);
  }
#undef GO
  return DRYFT_LAUNCH_CHECK();
}

template <typename E, int ROWS, int WAVES, bool GLU>
static int lines_by_rows(const void* x, int64_t x_stride, const void* w, void* y, int y_f32, int M, int N, int K, LateNorm<E> late,
                         Residual<E> residual, GateAct act, hipStream_t stream, const Beside<E>& beside = {}) {
  if constexpr (sizeof(E) == 4) {
    if (late.squares != nullptr) return launch_lines<E, ROWS, 1, WAVES, GLU, true>(x, x_stride, w, y, y_f32, M, N, K, late, residual, act, stream, beside);
    return launch_lines<E, ROWS, 1, WAVES, GLU, false>(x, x_stride, w, y, y_f32, M, N, K, late, residual, act, stream, beside);
  } else {
    if (late.squares != nullptr) {
      if (M <= 4) return launch_lines<E, ROWS, 1, WAVES, GLU, true>(x, x_stride, w, y, y_f32, M, N, K, late, residual, act, stream, beside);
      return launch_lines<E, ROWS, 2, WAVES, GLU, true>(x, x_stride, w, y, y_f32, M, N, K, late, residual, act, stream, beside);
    }
    if constexpr (!GLU) {
      if (beside.count > 0) {
        if (M <= 4) return launch_lines<E, ROWS, 1, WAVES, GLU, false, true>(x, x_stride, w, y, y_f32, M, N, K, late, residual, act, stream, beside);
        if (M <= 8) return launch_lines<E, ROWS, 2, WAVES, GLU, false, true>(x, x_stride, w, y, y_f32, M, N, K, late, residual, act, stream, beside);
        return launch_lines<E, ROWS, 4, WAVES, GLU, false, true>(x, x_stride, w, y, y_f32, M, N, K, late, residual, act, stream, beside);
      }
    }
    if (M <= 4) return launch_lines<E, ROWS, 1, WAVES, GLU, false>(x, x_stride, w, y, y_f32, M, N, K, late, residual, act, stream, beside);
    if (M <= 8) return launch_lines<E, ROWS, 2, WAVES, GLU, false>(x, x_stride, w, y, y_f32, M, N, K, late, residual, act, stream, beside);
    return launch_lines<E, ROWS, 4, WAVES, GLU, false>(x, x_stride, w, y, y_f32, M, N, K, late, residual, act, stream, beside);
  }
}

// Rows of a workgroup, and its waves: up to 3,072 outputs the fewest rows that leave every compute unit one workgroup (of eight
// waves, with registers for ten blocks on their way); 2,560 x 9,728 in 320 workgroups of eight rows instead of 256 of ten: 13.9 against
// 10.1 us, the units that get two of them work on alone. Beyond, four waves, several workgroups a unit, of as many rows as make
// their rounds fullest. Each workgroup reads the rows of x again: with more than four of them and a large matrix 20 weight rows
// share that (151,936 x 2,560 at 8 rows 132 us against 139 with 12; at 4 rows 121 either way; 10,240 x 5,120 at 8 18.9 against 20.4
// with 10; 5,120 x 8,192 16.8 against 16.6: the line). With little depth a wave has a block or two of K and a workgroup is mostly its
// ends: there bfloat16 takes 12 rows up to eight of x, the fewest workgroups (65,536 x 512 at one row 11.6 us, with the 8 that fill the rounds 17.9;
// 28,672 x 512 6.5 / 9.1; 32,000 x 1,024 11.6 / 13.6; up to K = 1,024; at 9 rows of x 8,192 x 512 5.2, with 8 4.1; 4,096 x 1,024 at four
// 3.8, with 8 3.5), and float32, whose sums fill its registers, 8, for the waves
// that fit beside one another (50,257 x 1,024 at one row 32.2, with 10 41.4; 17,408 x 1,536 18.8 / 22.7; up to K = 1,536).
#define LINES_LARGE ((int64_t)80 << 20)      // bytes of W
struct LinesShape {
  int rows, waves;
};
static LinesShape lines_shape(int M, int N, int64_t row_bytes, bool is_f32) {
  if (N <= 3072) return {N <= 1024 ? 4 : N <= 2048 ? 8 : N <= 2560 ? 10 : 12, 8};
  if (!is_f32 && M > 4 && N * row_bytes >= LINES_LARGE) return {20, 4};      // float32: no registers for so many sums
  if (M <= 8 && N > 4096 && row_bytes <= (is_f32 ? 6144 : 2048)) return {is_f32 ? 8 : 12, 4};
  int best = 12;
  int64_t least = INT64_MAX;
  for (int rows = 12; rows >= 8; rows -= 2) {
    const int64_t rounds = ((N + rows - 1) / rows + 255) / 256;
    if (rounds * rows < least) {
      least = rounds * rows;
      best = rows;
    }
  }
  return {best, 4};
}

// How many workgroups the product takes, and so how many rows of sums of squares it leaves.
DRYFT_API int dryft_gemm_lines_blocks(int M, int N, int K, int is_f32) {
  const int rows = lines_shape(M, N, (int64_t)K * (is_f32 ? 4 : 2), is_f32).rows;
  return (N + rows - 1) / rows;
}

template <typename E>
static bool lines_refuse(const void* x, int64_t x_stride, const void* w, int M, int K, const LateNorm<E>& late) {
  constexpr int V = Fragment<E>::VALUES;
  return M > (V == 8 ? LINES_ROWS : LINES_ROWS_F32) || K <= 0 || K % V || x_stride % V || (((uintptr_t)x | (uintptr_t)w) & 15) ||
         (late.squares != nullptr && (M > LATE_ROWS || late.count < 1 || late.count > LATE_MOST || late.weight == nullptr ||
                                      (((uintptr_t)late.squares | (uintptr_t)late.weight) & 15)));
}

template <typename E>
static int lines(const void* x, int64_t x_stride, const void* w, void* y, int y_f32, int M, int N, int K, const float* late_squares,
                 int late_count, float late_eps, const void* late_weight, void* residual_rows, float* squares, hipStream_t stream,
                 const Beside<E>& beside = {}) {
  if (M <= 0 || N <= 0) return 0;
  const LateNorm<E> late{late_squares, late_count, late_eps, (const E*)late_weight};
  const Residual<E> residual{(E*)residual_rows, squares};
  if (lines_refuse(x, x_stride, w, M, K, late) || (residual_rows != nullptr && (squares == nullptr || M > LATE_ROWS))) return -1;
  int outputs = N;
  for (int p = 0; p < beside.count; ++p) outputs += beside.n[p];
  const LinesShape shape = lines_shape(M, outputs, (int64_t)K * sizeof(E), sizeof(E) == 4);
#define LINES(ROWS, W) case ROWS + 32 * W: return lines_by_rows<E, ROWS, W, false>(x, x_stride, w, y, y_f32, M, N, K, late, residual, {}, stream, beside);
  switch (shape.rows + 32 * shape.waves) {
    LINES(4, 8) LINES(8, 8) LINES(10, 8) LINES(12, 8) LINES(8, 4) LINES(10, 4) LINES(12, 4)
    case 20 + 32 * 4:
      if constexpr (sizeof(E) == 2) return lines_by_rows<E, 20, 4, false>(x, x_stride, w, y, y_f32, M, N, K, late, residual, {}, stream, beside);
    default: return -1;
  }
#undef LINES
}

template <typename E>
static int lines_glu(const void* x, int64_t x_stride, const void* w, void* y, int M, int N, int K, const float* late_squares,
                     int late_count, float late_eps, const void* late_weight, GateAct act, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  const LateNorm<E> late{late_squares, late_count, late_eps, (const E*)late_weight};
  if (lines_refuse(x, x_stride, w, M, K, late) || act.limit < 0.f || (act.relu && act.limit > 0.f)) return -1;
  if (N <= 1024) return lines_by_rows<E, 8, 8, true>(x, x_stride, w, y, 0, M, N, K, late, {}, act, stream);
  return lines_by_rows<E, 16, 4, true>(x, x_stride, w, y, 0, M, N, K, late, {}, act, stream);
}

// M <= 16, K a multiple of 8, rows of x and W at 16-byte addresses. y as float (y_f32) or bfloat16, or with `residual` the sum
// residual[M, N] + y in place and squares[blocks][8] (M <= 8). late_squares: those of the product that left x (M <= 8).
DRYFT_API int dryft_gemm_lines_bf16(const void* x, int64_t x_stride, const void* w, void* y, int y_f32, int M, int N, int K,
                                    const float* late_squares, int late_count, float late_eps, const void* late_weight,
                                    void* residual, float* squares, hipStream_t stream) {
  return lines<bf16_t>(x, x_stride, w, y, y_f32, M, N, K, late_squares, late_count, late_eps, late_weight, residual, squares, stream);
}

// The products of x [M, K] with up to four matrices w[p] [n[p], K], each y[p] as float (y_f32[p]) or bfloat16, in one launch:
// gates, step sizes and the second mixer of two side by side, launches of 2.3 to 6 us and the gap before each, ride along with a
// layer's first product. Passes of 24 decoding steps of four sequences and their prompts, ms: barilix-w2048 (nine launches fewer a
// step) 20.8 -> 20.4, piralix-w2048 (two of its first six layers) 10.29 -> 10.14, fubinex-w2048 (four) 17.50 -> 17.26.
DRYFT_API int dryft_gemm_lines_beside_bf16(const void* x, int64_t x_stride, int M, int K, int count, const void* const* w, void* const* y,
                                           const int* n, const int* y_f32, hipStream_t stream) {
  if (count < 1 || count > 1 + LINES_BESIDE) return -1;
  Beside<bf16_t> beside;
  beside.count = count - 1;
  for (int p = 0; p < count; ++p)
    if (n[p] <= 0 || ((uintptr_t)w[p] & 15)) return -1;
  for (int p = 1; p < count; ++p) {
    beside.w[p - 1] = (const bf16_t*)w[p];
    beside.y[p - 1] = y[p];
    beside.n[p - 1] = n[p];
    beside.y_f32[p - 1] = y_f32[p];
  }
  return lines<bf16_t>(x, x_stride, w[0], y[0], y_f32[0], M, n[0], K, nullptr, 0, 0.f, nullptr, nullptr, nullptr, stream, beside);
}

// The same in float32: M <= 4, K a multiple of 4. Us at 1 / 4 rows, against the kernels of gemm_f32.hip: 4,096 x 1,024 5.6 / 5.5 (6.0 /
// 6.7), 1,024 x 3,072 4.9 / 5.1 (5.8 / 6.2), 151,936 x 1,024 95 / 95 (104 / 120), 6,144 x 2,560 13.3 / 13.6 (13.4 / 18.5), 2,560 x 9,728
// 20.7 / 20.9 (32 / 39), 3,072 gated outputs of 1,024 7.4 / 7.6 (9.6 / 10.3). At 8 rows the sums of two groups of four leave one
// workgroup a unit: 151,936 x 1,024 217 us against 157.
DRYFT_API int dryft_gemm_lines_f32(const void* x, int64_t x_stride, const void* w, void* y, int M, int N, int K,
                                   const float* late_squares, int late_count, float late_eps, const void* late_weight,
                                   void* residual, float* squares, hipStream_t stream) {
  return lines<float>(x, x_stride, w, y, 1, M, N, K, late_squares, late_count, late_eps, late_weight, residual, squares, stream);
}

// y[M,N] = the gated unit of x . Wg^T and x . Wu^T with W = [Wg; Wu] of 2N rows. Up to 1,024 outputs four a workgroup of eight waves,
// beyond eight a workgroup of four. Us at 1 / 4 / 8 / 16 rows against the panel product (gemm.hip): 9,728 outputs of K 2,560 17.4 /
// 17.2 / 18.3 / 21.4 (19.7 / 19.9 / 20.0 / 20.2), 12,288 of 4,096 33.0 / 32.4 / 33.0 / 37.2 (37.7 / 36.2 / 36.4 / 36.5), 8,192 of 2,048
// 12.2 / 12.4 / 14.0 / 16.4 (12.7 / 12.7 / 12.7 / 12.8), 4,096 of 2,048 7.4 / 7.7 / 8.0 / 9.1 (9.3 / 9.3 / 9.5 / 9.7); 3,072 of 1,024 4.5 / 4.6
// / 4.9 / 5.7 (6.3 / 5.9 / - / 6.1), and against a kernel that took each operand's rows 32 bytes at a time 1,024 of 2,048 4.0 / 4.1 / 4.2 / 4.7
// (5.1 / 5.4 / 5.9 / 6.7), 512 of 2,048 3.5 / 3.6 / 3.8 / 4.4 (4.7 / 5.1 / 5.4 / 6.1): `gemm_few_glu_ok` in ops.py draws the line.
DRYFT_API int dryft_gemm_lines_glu_bf16(const void* x, int64_t x_stride, const void* w, void* y, int M, int N, int K,
                                        const float* late_squares, int late_count, float late_eps, const void* late_weight, int relu,
                                        float limit, float alpha, hipStream_t stream) {
  GateAct act;
  act.relu = relu;
  act.limit = limit;
  act.alpha = alpha;
  return lines_glu<bf16_t>(x, x_stride, w, y, M, N, K, late_squares, late_count, late_eps, late_weight, act, stream);
}

// silu(x . Wg^T) * (x . Wu^T) in float32: M <= 4, K a multiple of 4
DRYFT_API int dryft_gemm_lines_swiglu_f32(const void* x, int64_t x_stride, const void* w, void* y, int M, int N, int K,
                                          const float* late_squares, int late_count, float late_eps, const void* late_weight,
                                          hipStream_t stream) {
  return lines_glu<float>(x, x_stride, w, y, M, N, K, late_squares, late_count, late_eps, late_weight, {}, stream);
}
