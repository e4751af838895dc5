// One token of a sequence through a matrix state [D, P] a head, for steps in which every sequence has one row (decoding): the delta
// rule, the state-space recurrence and the matrix memory of delta.hip, ssm.hip and mlstm.hip, with their formulas.
//
// A workgroup takes one (sequence, head); a thread keeps four neighbouring columns of the state rows rg, rg + RG, ..., so that the
// state goes by in whole lines and every load of the step is out before anything waits. Column sums meet in LDS. The read-outs of the
// delta rule and the matrix memory are normed per head and gated in the same launch.
// Bound by trips to memory one after the other (the sequence's slot, its state and operands) and the launch's ends, not by the
// state's bytes. The kernels that walk a sequence row by row keep a column in neighbouring lanes (a quarter of a line a load) and
// stage eight rows' operands for the one there is. Delta rule with its read-out, 16 heads of 128 x 128, 4 / 16 / 64 / 256 sequences: 7.0,
// 9.3, 28 and 102 us (5.3 TB/s), where walk and read-out took 12.5, 24, 51 and 201; state-space, 32 heads of 128 x 64: 5.4, 9.1, 27 and
// 97 us, where the walk took 9.4, 20, 72 and 303; matrix memory with its read-out, 8 heads of
// 128 x 256: 7.9, 9.9, 28 and 102 us, where walk and read-out took 10.9, 18, 56 and 212.
#pragma once
#include "common.h"

#define TOKEN_MAX_DIM 256

enum TokenKind { TOKEN_SSM, TOKEN_DELTA, TOKEN_MEMORY };

struct TokenStep {
  int64_t stride;                  // of a row of q | k | v (C | B | x)
  int q_col, k_col, v_col;
  const float* gates;              // [rows, gate_stride]: a_col + head the decay's input, b_col + head the delta rule's beta;
                                   // the memory's log input and log forget gates
  int64_t gate_stride;
  int a_col, b_col;
  const float *dt_bias, *a_log, *d_skip;                           // the memory: the gates' two biases
  const int *seq_slot, *cu_rows, *q_len;
  float* state;
  int H, G, D, P;
  float q_scale, unit_eps;
  int write_state;
  int64_t out_gate_stride;         // the normed read-outs: gate of a row, weight [H P], eps
  const float* weight;
  float eps;
  float cap;                       // the memory: cap of its gates, normaliser [slots, H, copies, D] and maximum [slots, H, copies]
  float *normaliser, *maximum;
  int copies;
};

template <typename T, int KIND, int THREADS, int NR>
__global__ __launch_bounds__(THREADS) void token_step_kernel(const T* __restrict__ x, const T* __restrict__ out_gate,
                                                                   void* __restrict__ out, TokenStep a) {
  constexpr int WAVES = THREADS / WAVE;
  constexpr bool DELTA = KIND == TOKEN_DELTA, MEMORY = KIND == TOKEN_MEMORY, NORMED = DELTA || MEMORY;
  __shared__ float sq[TOKEN_MAX_DIM], sk[TOKEN_MAX_DIM], squares[2][TOKEN_MAX_DIM / WAVE], red[WAVES][TOKEN_MAX_DIM];
  __shared__ __attribute__((aligned(16))) float su[TOKEN_MAX_DIM];
  const int seq = blockIdx.x, head = blockIdx.y, tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
  const int D = a.D, P = a.P, slot = a.seq_slot[seq];
  const int64_t row = a.cu_rows[seq];
  if (a.q_len[seq] <= 0) return;
  if (slot < 0) {                                          // sits out: zeros where the read-out's norm would have left them
    if (NORMED && tid < P) store_from_float((T*)out + (row * a.H + head) * P + tid, 0.f);
    return;
  }
  const int C = P / 4, c = tid % C, rg = tid / C, RG = THREADS / C;      // C: 8, 16, 32 or 64
  float* at = a.state + (((int64_t)slot * a.H + head) * D + rg) * P + 4 * c;
  vf4 S[NR];
#pragma unroll
  for (int j = 0; j < NR; ++j) S[j] = rg + j * RG < D ? *(const vf4*)(at + (int64_t)j * RG * P) : vf4{0.f, 0.f, 0.f, 0.f};
  const T* p = x + row * a.stride;
  const int group = head / (a.H / a.G);
  const float k = tid < D ? load_as_float(p + a.k_col + group * D + tid) : 0.f;
  const float q = tid < D ? load_as_float(p + a.q_col + group * D + tid) : 0.f;
  const float v = tid < P ? load_as_float(p + a.v_col + head * P + tid) : 0.f;
  const float z = a.gates[row * a.gate_stride + a.a_col + head] + a.dt_bias[head], rate = a.a_log[head];
  const float b = NORMED ? a.gates[row * a.gate_stride + a.b_col + head] : a.d_skip[head];
  const float gate = NORMED && tid < P ? load_as_float(out_gate + row * a.out_gate_stride + head * P + tid) : 0.f;
  const float weight = NORMED && tid < P ? a.weight[head * P + tid] : 0.f;
  float g, take, peak = 0.f;                               // the state's decay, what the token's outer product weighs
  if constexpr (MEMORY) {
    const int64_t at_n = ((int64_t)slot * a.H + head) * a.copies;        // every copy holds the same: the first is read
    const float n = tid < D ? a.normaliser[at_n * D + tid] : 0.f, m = a.maximum[at_n];
    const float gi = a.cap * tanhf(z / a.cap), f = a.cap * tanhf((b + rate) / a.cap);
    const float gf = fminf(f, 0.f) - log1pf(expf(-fabsf(f)));
    peak = fmaxf(gf + m, gi);
    g = expf(gf + m - peak);
    take = expf(gi - peak);
    const float n_new = g * n + k * take;
    const float nq = wave_sum(tid < D ? n_new * (q * a.q_scale) : 0.f);
    if (wave < TOKEN_MAX_DIM / WAVE && lane == 0) squares[1][wave] = nq;
    __syncthreads();                                       // the first copy has been read by every wave
    if (a.write_state) {
      for (int y = 0; y < a.copies; ++y) {
        if (tid < D) a.normaliser[(at_n + y) * D + tid] = n_new;
        if (tid == 0) a.maximum[at_n + y] = peak;
      }
    }
  } else {
    const float dt = z > 20.f ? z : log1pf(expf(z));
    g = expf(-expf(rate) * dt);
    take = dt;
  }
  if (DELTA && wave < TOKEN_MAX_DIM / WAVE) {
    const float kk = wave_sum(k * k), qq = wave_sum(q * q);
    if (lane == 0) { squares[0][wave] = kk; squares[1][wave] = qq; }
  }
  if (tid < D) { sk[tid] = k; sq[tid] = MEMORY ? q * a.q_scale : q; }
  if (!DELTA && tid < P) su[tid] = take * v;
  __syncthreads();
  float k_unit = 1.f, q_unit = 1.f;
  if (DELTA) {
    k_unit = rsqrtf((squares[0][0] + squares[0][1]) + (squares[0][2] + squares[0][3]) + a.unit_eps);
    q_unit = rsqrtf((squares[1][0] + squares[1][1]) + (squares[1][2] + squares[1][3]) + a.unit_eps) * a.q_scale;
  }
  // a column's sum over the wave's rows in the lanes below C, then over the waves in the threads below P
  auto column_sum = [&](vf4 part) {
#pragma unroll
    for (int o = 8; o < WAVE; o <<= 1) {
      if (o < C) continue;
#pragma unroll
      for (int u = 0; u < 4; ++u) part[u] += __shfl_xor(part[u], o, WAVE);
    }
    if (lane < C) {
#pragma unroll
      for (int u = 0; u < 4; ++u) red[wave][4 * c + u] = part[u];
    }
    __syncthreads();
    float sum = 0.f;
    if (tid < P) {
#pragma unroll
      for (int w = 0; w < WAVES; ++w) sum += red[w][tid];
    }
    return sum;
  };
  if (DELTA) {
    vf4 old = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NR; ++j) old += S[j] * (rg + j * RG < D ? sk[rg + j * RG] * k_unit : 0.f);
    const float read = column_sum(old);
    if (tid < P) su[tid] = 1.f / (1.f + expf(-b)) * (v - g * read);
    __syncthreads();
  }
  const vf4 u = *(const vf4*)(su + 4 * c);
  vf4 res = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    const int r = rg + j * RG;
    if (r >= D) continue;
    S[j] = g * S[j] + sk[r] * k_unit * u;
    res += S[j] * (sq[r] * q_unit);
    if (a.write_state) *(vf4*)(at + (int64_t)j * RG * P) = S[j];
  }
  float o = column_sum(res);
  if constexpr (!NORMED) {
    if (tid < P) ((float*)out)[(row * a.H + head) * P + tid] = o + b * v;
    return;
  }
  if (MEMORY) o /= fmaxf(fabsf((squares[1][0] + squares[1][1]) + (squares[1][2] + squares[1][3])), expf(-peak)) + 1e-6f;
  const float oo = wave_sum(tid < P ? o * o : 0.f);
  if (wave < TOKEN_MAX_DIM / WAVE && lane == 0) squares[0][wave] = oo;
  __syncthreads();
  const float mean = ((squares[0][0] + squares[0][1]) + (squares[0][2] + squares[0][3])) / (float)P;
  const float gated = (DELTA ? gate : 1.f) / (1.f + expf(-gate));
  if (tid < P) store_from_float((T*)out + (row * a.H + head) * P + tid, o * (1.f / sqrtf(mean + a.eps)) * weight * gated);
}

// -2: sizes that the kernel does not take (P of 32, 64, 128 and 256, state at 16-byte addresses).
template <int KIND>
static int token_step_run(const void* x, const void* out_gate, void* out, const TokenStep& a, int n_seqs, int is_f32, hipStream_t stream) {
  if (n_seqs <= 0) return 0;
  if (a.H <= 0 || a.G <= 0 || a.H % a.G || a.D <= 0) return -1;
  if (a.D > TOKEN_MAX_DIM || (a.P != 32 && a.P != 64 && a.P != 128 && a.P != 256) || ((uintptr_t)a.state & 15) || a.H > 65535) return -2;
  // rows a thread of 256 would take: with more than 4 each, 1,024 threads take a quarter of them
  // (2 to 16). 8 heads of a 64 x 32 state for 1 and 256 sequences: 3.9 and 8.7 us with 256 threads, 4.4 and 17.8 with 1,024; 32 heads of
  // 128 x 64 need the loads of 1,024 in flight.
  const int RG = 256 / (a.P / 4), per = (a.D + RG - 1) / RG;
#define TOKEN(TT, THREADS, NN)                                                                                                  \
  hipLaunchKernelGGL((token_step_kernel<TT, KIND, THREADS, NN>), dim3(n_seqs, a.H), dim3(THREADS), 0, stream, (const TT*)x, \
                     (const TT*)out_gate, out, a)
#define TOKENS(TT)                                             \
  if (per <= 1) TOKEN(TT, 256, 1);                             \
  else if (per <= 4) TOKEN(TT, 256, 4);                        \
  else if (per <= 8) TOKEN(TT, 1024, 2);                       \
  else if (per <= 16) TOKEN(TT, 1024, 4);                      \
  else if (per <= 32) TOKEN(TT, 1024, 8);                      \
  else TOKEN(TT, 1024, 16)
  if (is_f32) {
    TOKENS(float);
  } else {
    TOKENS(bf16_t);
  }
#undef TOKENS
#undef TOKEN
  return DRYFT_LAUNCH_CHECK();
}
