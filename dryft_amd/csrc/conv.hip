// A short causal convolution over time on every channel of a projection, with the sequence's last inputs kept as
// state so that a prompt, a portion of one and a single token are the same code.
//
//   y[t, c] = act( sum_j w[c, j] * u[t - taps + 1 + j, c] + b[c] ),      u = projection (+ its own bias)
//
// with zeros before a sequence's start. The inputs of the `taps - 1` positions before this step's rows come from
// `tail [slots, taps - 1, C]` (float32, zero for a sequence that starts); a second kernel moves the tail on once
// every row has read it. All arithmetic is float; y is rounded once.
#include "common.h"

#define CONV_MAX_TAPS 16

template <typename T>
__global__ __launch_bounds__(256) void causal_conv_kernel(const T* __restrict__ u, int64_t u_stride, int col,
                                                          const float* __restrict__ in_bias,
                                                          const float* __restrict__ w, const float* __restrict__ out_bias,
                                                          int taps, int act, const int* __restrict__ row_slot,
                                                          const int* __restrict__ row_seq,
                                                          const int* __restrict__ row_pos,
                                                          const int* __restrict__ seq_start,
                                                          const float* __restrict__ tail, T* __restrict__ out, int C) {
  const int64_t row = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int slot = row_slot[row];
  if (slot < 0) {
    store_from_float(out + row * C + c, 0.f);
    return;
  }
  const int pos = row_pos[row], start = seq_start[row_seq[row]];
  const float ib = in_bias ? in_bias[c] : 0.f;
  float acc = out_bias ? out_bias[c] : 0.f;
  for (int j = 0; j < taps; ++j) {
    const int d = taps - 1 - j, p = pos - d;
    float v = 0.f;
    if (p >= start) v = load_as_float(u + (row - d) * u_stride + col + c) + ib;
    else if (p >= 0 && tail != nullptr) v = tail[((int64_t)slot * (taps - 1) + (p - start + taps - 1)) * C + c];
    acc += w[(int64_t)c * taps + j] * v;
  }
  if (act == 1) acc = acc / (1.f + expf(-acc));
  store_from_float(out + row * C + c, acc);
}

// One row of eight neighbouring channels, read and written 16 bytes at a time, with the weights tap by tap (`w_t [taps, C]`):
// for inputs, outputs and tails whose rows start at multiples of 8 channels.
template <typename T>
__device__ __forceinline__ void conv_row_of_eight(int64_t row, int c, const T* __restrict__ u, int64_t u_stride, int col,
                                                  const float* __restrict__ in_bias, const float* __restrict__ w_t,
                                                  const float* __restrict__ out_bias, int taps, int act,
                                                  const int* __restrict__ row_slot, const int* __restrict__ row_seq,
                                                  const int* __restrict__ row_pos, const int* __restrict__ seq_start,
                                                  const float* __restrict__ tail, T* __restrict__ out, int C) {
  const int slot = row_slot[row];
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (slot < 0) {
    store8_from_float(out + row * C + c, acc);
    return;
  }
  const int pos = row_pos[row], start = seq_start[row_seq[row]];
  float ib[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (in_bias) load8_as_float(in_bias + c, ib);
  if (out_bias) load8_as_float(out_bias + c, acc);
  for (int j = 0; j < taps; ++j) {
    const int d = taps - 1 - j, p = pos - d;
    float v[8], wj[8];
    if (p >= start) {
      load8_as_float(u + (row - d) * u_stride + col + c, v);
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] += ib[i];
    } else if (p >= 0 && tail != nullptr) {
      load8_as_float(tail + ((int64_t)slot * (taps - 1) + (p - start + taps - 1)) * C + c, v);
    } else {
      continue;
    }
    load8_as_float(w_t + (int64_t)j * C + c, wj);
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] += wj[i] * v[i];
  }
  if (act == 1) {
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = acc[i] / (1.f + expf(-acc[i]));
  }
  store8_from_float(out + row * C + c, acc);
}

// A thread a row of eight channels.
template <typename T>
__global__ __launch_bounds__(256) void causal_conv_vec_kernel(const T* __restrict__ u, int64_t u_stride, int col,
                                                              const float* __restrict__ in_bias,
                                                              const float* __restrict__ w_t,
                                                              const float* __restrict__ out_bias, int taps, int act,
                                                              const int* __restrict__ row_slot,
                                                              const int* __restrict__ row_seq,
                                                              const int* __restrict__ row_pos,
                                                              const int* __restrict__ seq_start,
                                                              const float* __restrict__ tail, T* __restrict__ out, int C) {
  const int64_t row = blockIdx.x;
  const int c = (blockIdx.y * blockDim.x + threadIdx.x) * 8;
  if (c >= C) return;
  conv_row_of_eight(row, c, u, u_stride, col, in_bias, w_t, out_bias, taps, act, row_slot, row_seq, row_pos, seq_start, tail, out, C);
}

// R rows of eight channels a thread: where they are neighbours of one sequence with all the inputs they need among this step's rows,
// R + TAPS - 1 loads go out together instead of R x TAPS, and the weights are read once; other runs of rows go one by one. Sums in the
// same order, so the same bits.
// Bound by bytes, of which a row a thread asks TAPS times over, behind a chain of facts and taps. us a row a thread / four rows, bfloat16,
// 4 taps, one sequence: 2,048 x 2,048 11.2 / 9.2, 2,048 x 4,096 19.6 / 14.5, 5,099 x 4,096 38.4 / 27.2, x 8,192 70.7 / 47.3 (3.5 TB/s);
// float32 5,099 x 8,192 136 / 79. Eight rows: 9.2 to 15.6, 14.5 to 19.2, 27.2 to 28.1, 47.3 to 46.1: too few waves but for the largest.
template <typename T, int TAPS, int R>
__global__ __launch_bounds__(256) void causal_conv_rows_kernel(const T* __restrict__ u, int64_t u_stride, int col,
                                                               const float* __restrict__ in_bias,
                                                               const float* __restrict__ w_t,
                                                               const float* __restrict__ out_bias, int act,
                                                               const int* __restrict__ row_slot,
                                                               const int* __restrict__ row_seq,
                                                               const int* __restrict__ row_pos,
                                                               const int* __restrict__ seq_start,
                                                               const float* __restrict__ tail, T* __restrict__ out, int n_rows, int C) {
  const int64_t r0 = (int64_t)blockIdx.x * R;
  const int c = (blockIdx.y * blockDim.x + threadIdx.x) * 8;
  if (c >= C) return;
  bool together = r0 + R <= n_rows;
  if (together) {
    const int seq = row_seq[r0], pos = row_pos[r0];
    bool same = true;
#pragma unroll
    for (int i = 0; i < R; ++i) same &= row_slot[r0 + i] >= 0 && row_seq[r0 + i] == seq && row_pos[r0 + i] == pos + i;
    together = same && pos - (TAPS - 1) >= seq_start[seq];
  }
  if (!together) {
    for (int64_t row = r0; row < r0 + R && row < n_rows; ++row)
      conv_row_of_eight(row, c, u, u_stride, col, in_bias, w_t, out_bias, TAPS, act, row_slot, row_seq, row_pos, seq_start, tail, out, C);
    return;
  }
  float wj[TAPS][8], ib[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, ob[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  float v[R + TAPS - 1][8];
#pragma unroll
  for (int i = 0; i < R + TAPS - 1; ++i) load8_as_float(u + (r0 + i - (TAPS - 1)) * u_stride + col + c, v[i]);
#pragma unroll
  for (int j = 0; j < TAPS; ++j) load8_as_float(w_t + (int64_t)j * C + c, wj[j]);
  if (in_bias) load8_as_float(in_bias + c, ib);
  if (out_bias) load8_as_float(out_bias + c, ob);
#pragma unroll
  for (int i = 0; i < R + TAPS - 1; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) v[i][e] += ib[e];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      acc[e] = ob[e];
#pragma unroll
      for (int j = 0; j < TAPS; ++j) acc[e] += wj[j][e] * v[i + j][e];
      if (act == 1) acc[e] = acc[e] / (1.f + expf(-acc[e]));
    }
    store8_from_float(out + (r0 + i) * C + c, acc);
  }
}

// The tail after the step: the last taps - 1 inputs of each sequence, from this step's rows and, where the step
// brought fewer, from the tail before. A thread owns one (sequence, channel) and reads everything before it writes.
template <typename T>
__global__ __launch_bounds__(256) void conv_tail_kernel(const T* __restrict__ u, int64_t u_stride, int col,
                                                        const float* __restrict__ in_bias, int taps,
                                                        const int* __restrict__ seq_slot,
                                                        const int* __restrict__ cu_rows, const int* __restrict__ q_len,
                                                        float* __restrict__ tail, int C) {
  const int seq = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  const int slot = seq_slot[seq], q = q_len[seq];
  if (c >= C || slot < 0 || q <= 0) return;
  const int keep = taps - 1;
  const int64_t first = cu_rows[seq];
  const float ib = in_bias ? in_bias[c] : 0.f;
  float* mine = tail + (int64_t)slot * keep * C + c;
  float v[CONV_MAX_TAPS];
#pragma unroll
  for (int j = 0; j < CONV_MAX_TAPS - 1; ++j) {
    if (j < keep) {
      const int r = q - keep + j;             // the step's row that lands in place j, if it has one
      v[j] = r >= 0 ? load_as_float(u + (first + r) * u_stride + col + c) + ib : mine[(int64_t)(j + q) * C];
    }
  }
#pragma unroll
  for (int j = 0; j < CONV_MAX_TAPS - 1; ++j)
    if (j < keep) mine[(int64_t)j * C] = v[j];
}

// Both for steps that bring each sequence one row (decoding): every earlier input lies in the tail, and the thread that
// reads a channel of it is the only one to do so, so it moves the tail on itself. All loads are asked for before the first
// sum; sums in the order of the kernels above. Such a step is bound by its launches and the trips to memory behind each:
// 4 rows of 10,240 to 16,384 channels, 4 taps, in a step: 4.4 us, in two launches 4.9 and 4.8. In a chain, 10,240 channels at 4 /
// 32 / 64 / 256 rows 3.5 / 5.0 / 7.3 / 21.3 us, in two launches (from 32 rows on eight channels a thread) 5.5 / 8.6 / 11.0 / 29.3.
template <typename T>
__global__ __launch_bounds__(256) void conv_step_kernel(const T* __restrict__ u, int64_t u_stride, int col,
                                                        const float* __restrict__ in_bias, const float* __restrict__ w,
                                                        int w_channel, int w_tap, const float* __restrict__ out_bias, int taps,
                                                        int act, const int* __restrict__ row_slot, const int* __restrict__ row_pos,
                                                        float* __restrict__ tail, T* __restrict__ out, int C) {
  const int64_t row = blockIdx.x;
  const int c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  float wj[CONV_MAX_TAPS], v[CONV_MAX_TAPS];
#pragma unroll
  for (int j = 0; j < CONV_MAX_TAPS; ++j)
    if (j < taps) wj[j] = w[(int64_t)c * w_channel + (int64_t)j * w_tap];
  const float now = load_as_float(u + row * u_stride + col + c) + (in_bias ? in_bias[c] : 0.f);
  float acc = out_bias ? out_bias[c] : 0.f;
  const int slot = row_slot[row], pos = row_pos[row], keep = taps - 1;
  if (slot < 0) {
    store_from_float(out + row * C + c, 0.f);
    return;
  }
  float* mine = tail + (int64_t)slot * keep * C + c;
#pragma unroll
  for (int j = 0; j < CONV_MAX_TAPS; ++j)
    if (j < taps) v[j] = j < keep ? mine[(int64_t)j * C] : now;
#pragma unroll
  for (int j = 0; j < CONV_MAX_TAPS; ++j)
    if (j < taps) {
      acc += wj[j] * (pos - (keep - j) >= 0 ? v[j] : 0.f);
      if (j > 0) mine[(int64_t)(j - 1) * C] = v[j];
    }
  if (act == 1) acc = acc / (1.f + expf(-acc));
  store_from_float(out + row * C + c, acc);
}

DRYFT_API int dryft_conv_max_taps() { return CONV_MAX_TAPS; }

DRYFT_API int dryft_causal_conv(const void* u, int64_t u_stride, int col, const float* in_bias, const float* w,
                                const float* w_t, const float* out_bias, int taps, int act, const int* row_slot,
                                const int* row_seq, const int* row_pos, const int* seq_start, const float* tail, void* out,
                                int n_rows, int n_seqs, int C, int is_f32, hipStream_t stream) {
  if (n_rows <= 0) return 0;
  if (taps < 1 || taps > CONV_MAX_TAPS || C <= 0 || (taps > 1 && tail == nullptr)) return -1;
  auto aligned = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  // steps of few rows keep the kernel of a channel a thread: eight times the threads for the same few loads each
  if (n_rows >= 32 && w_t != nullptr && C % 8 == 0 && col % 8 == 0 && u_stride % 8 == 0 && aligned(u) && aligned(out) && aligned(w_t) &&
      aligned(tail) && aligned(in_bias) && aligned(out_bias)) {
    const int across = (C / 8 + 255) / 256;
    // Four rows a thread where that leaves enough waves, in loads of a row a thread: 16 Mi values. Below, us a row a thread / four: 616 x 4,096
    // of 4 taps 7.7 / 9.8, 700 x 8,192 of 2 taps 10.8 / 11.4; on the line 2,048 x 2,048 of 4 taps 11.2 / 9.2, 616 x 8,192 13.6 / 12.6. And 16 rows
    // a sequence or more, since runs across a sequence's start go row by row: 5,100 x 4,096 in sequences of 17 36.1 / 32.2, of 5 32.4 / 37.3.
    if (taps >= 2 && taps <= 4 && (int64_t)n_rows * C * taps >= (16 << 20) && n_rows / 16 >= n_seqs) {
#define CONV_ROWS(TT, TAPS)                                                                                                \
  hipLaunchKernelGGL((causal_conv_rows_kernel<TT, TAPS, 4>), dim3((n_rows + 3) / 4, across), dim3(256), 0, stream, (const TT*)u, \
                     u_stride, col, in_bias, w_t, out_bias, act, row_slot, row_seq, row_pos, seq_start, tail, (TT*)out, n_rows, C)
      if (is_f32) {
        if (taps == 2) CONV_ROWS(float, 2);
        else if (taps == 3) CONV_ROWS(float, 3);
        else CONV_ROWS(float, 4);
      } else {
        if (taps == 2) CONV_ROWS(bf16_t, 2);
        else if (taps == 3) CONV_ROWS(bf16_t, 3);
        else CONV_ROWS(bf16_t, 4);
      }
#undef CONV_ROWS
      return DRYFT_LAUNCH_CHECK();
    }
    dim3 grid(n_rows, across), block(256);
    if (is_f32)
      hipLaunchKernelGGL(causal_conv_vec_kernel<float>, grid, block, 0, stream, (const float*)u, u_stride, col, in_bias,
                         w_t, out_bias, taps, act, row_slot, row_seq, row_pos, seq_start, tail, (float*)out, C);
    else
      hipLaunchKernelGGL(causal_conv_vec_kernel<bf16_t>, grid, block, 0, stream, (const bf16_t*)u, u_stride, col, in_bias,
                         w_t, out_bias, taps, act, row_slot, row_seq, row_pos, seq_start, tail, (bf16_t*)out, C);
    return DRYFT_LAUNCH_CHECK();
  }
  dim3 grid(n_rows, (C + 255) / 256), block(256);
  if (is_f32)
    hipLaunchKernelGGL(causal_conv_kernel<float>, grid, block, 0, stream, (const float*)u, u_stride, col, in_bias, w,
                       out_bias, taps, act, row_slot, row_seq, row_pos, seq_start, tail, (float*)out, C);
  else
    hipLaunchKernelGGL(causal_conv_kernel<bf16_t>, grid, block, 0, stream, (const bf16_t*)u, u_stride, col, in_bias, w,
                       out_bias, taps, act, row_slot, row_seq, row_pos, seq_start, tail, (bf16_t*)out, C);
  return DRYFT_LAUNCH_CHECK();
}

DRYFT_API int dryft_conv_tail(const void* u, int64_t u_stride, int col, const float* in_bias, int taps,
                              const int* seq_slot, const int* cu_rows, const int* q_len, float* tail, int n_seqs, int C,
                              int is_f32, hipStream_t stream) {
  if (n_seqs <= 0 || taps <= 1) return 0;
  if (taps > CONV_MAX_TAPS || C <= 0 || tail == nullptr) return -1;
  dim3 grid(n_seqs, (C + 255) / 256), block(256);
  if (is_f32)
    hipLaunchKernelGGL(conv_tail_kernel<float>, grid, block, 0, stream, (const float*)u, u_stride, col, in_bias, taps,
                       seq_slot, cu_rows, q_len, tail, C);
  else
    hipLaunchKernelGGL(conv_tail_kernel<bf16_t>, grid, block, 0, stream, (const bf16_t*)u, u_stride, col, in_bias, taps,
                       seq_slot, cu_rows, q_len, tail, C);
  return DRYFT_LAUNCH_CHECK();
}

DRYFT_API int dryft_conv_step(const void* u, int64_t u_stride, int col, const float* in_bias, const float* w, const float* w_t,
                              const float* out_bias, int taps, int act, const int* row_slot, const int* row_pos, float* tail,
                              void* out, int n_rows, int C, int is_f32, hipStream_t stream) {
  if (n_rows <= 0) return 0;
  if (taps < 2 || taps > CONV_MAX_TAPS || C <= 0 || tail == nullptr) return -1;
  dim3 grid(n_rows, (C + 255) / 256), block(256);
  const float* weights = w_t != nullptr ? w_t : w;             // tap by tap: neighbouring threads read neighbouring words
  const int w_channel = w_t != nullptr ? 1 : taps, w_tap = w_t != nullptr ? C : 1;
  if (is_f32)
    hipLaunchKernelGGL(conv_step_kernel<float>, grid, block, 0, stream, (const float*)u, u_stride, col, in_bias, weights, w_channel,
                       w_tap, out_bias, taps, act, row_slot, row_pos, tail, (float*)out, C);
  else
    hipLaunchKernelGGL(conv_step_kernel<bf16_t>, grid, block, 0, stream, (const bf16_t*)u, u_stride, col, in_bias, weights,
                       w_channel, w_tap, out_bias, taps, act, row_slot, row_pos, tail, (bf16_t*)out, C);
  return DRYFT_LAUNCH_CHECK();
}
