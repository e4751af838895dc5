// Recurrences with a matrix state per head, sixteen tokens at a time on the matrix cores in 32 bits
// (v_mfma_f32_16x16x4_f32: 32-bit factors, 32-bit sums). Per token, S being D x P:
//
//   delta rule:    S <- g S;   u = beta (v - S^T k);   S <- S + k u^T;   o = S^T q
//   state space:   S <- g S;   u = dt v;               S <- S + k u^T;   o = S^T q + d v       (k = B, q = C, v = x)
//
// With S the state that enters the chunk, p_i the product of the decays up to token i and m_ij that of the tokens after
// j up to i (all at most 1):
//
//   (I + L) U = beta (V - p K S),   L_ij = beta_i m_ij (k_i . k_j) for j < i
//   O = p Q S + A U,                A_ij = m_ij (q_i . k_j) for j <= i
//   S <- p_15 S + K^T (m_15 U)
//
// A workgroup owns 32 or 64 value columns of a head of a sequence and walks the sequence's rows of the step in order. Its
// owners, a wave for 16 columns, hold their part of S in the accumulators for the whole walk: lane (c, g) holds rows
// 4 g + r of every 16 rows of S at column c, which is also where the second operand of the next product wants its values
// if the sum over D (or over the tokens) is taken in the order 4 g + r, so that neither S nor U ever moves between lanes.
// Four helpers bring rows in and form L and A (each half of D into a plane of its own), one wave the decays and
// (I + L)^-1 by forward substitution. All meet at one barrier a chunk, which leaves loads from memory in flight:
//
//   owners:   U, O and the new S of chunk n, then K S and Q S of n + 1
//   helpers:  rows of n + 3 into LDS, L and A of n + 2              the last wave: decays of n + 3, (I + L)^-1 of n + 1
//
// Decays are exponents summed in 64 bits, m_ij the exp of a difference; unit vectors keep their direction exact (only a
// power of two is taken in), the rest of 1 / length enters with the factors of a row. Against 64 bits the error is that of
// a walk row by row where the state forgets within some rows (1.1e-7 to 1.5e-7 of the outputs' size, 1.2e-7 to 1.4e-7 row
// by row) and a third of it where it keeps hundreds of rows (3.4e-7, 1.15e-6).
//
// What bounds it is the owners' chain: 104 matrix instructions of 32 cycles for 16 tokens of the delta rule at D = 128
// (1.4 us), 68 for the state space (0.9 us); a chunk takes 2.5 and 1.9 us. With two barriers and helpers one chunk ahead it
// took 3.8 (delta rule): inverse, decays and products of the next chunk stood in the owners' way. 16 heads of
// 128 x 128, 5,099 rows of four sequences: 1,498 us as segments row by row, 335 us here; state space, 32 heads of
// 128 x 64: 817 and 254 us.
#pragma once
#include "common.h"

#define CW_TOKENS 16
#define CW_RING 4                 // chunks in LDS: one is applied, one read out, one multiplied with itself, one brought in
typedef __attribute__((ext_vector_type(4))) float cw_f4;
__device__ __forceinline__ cw_f4 cw_mfma(float a, float b, cw_f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
// all waves' LDS traffic before this is done; loads from memory into registers stay in flight
__device__ __forceinline__ void cw_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ float cw_softplus(float z) { return z > 20.f ? z : log1pf(expf(z)); }

// Eight neighbouring values as they lie in memory: what is asked for stays raw until it is used, so that a wave waits for
// it there; rows and columns beyond the end are asked for at a valid place and replaced by zeros then.
__device__ __forceinline__ void cw_raw8(const bf16_t* p, vu4 (&v)[2]) { v[0] = *(const vu4*)p; }
__device__ __forceinline__ void cw_raw8(const float* p, vu4 (&v)[2]) { v[0] = *(const vu4*)p; v[1] = *(const vu4*)(p + 4); }
template <typename T>
__device__ __forceinline__ float cw_value(const vu4 (&v)[2], int j) {
  if (sizeof(T) == 4) return __uint_as_float(v[j / 4][j % 4]);
  return __uint_as_float(j & 1 ? v[0][j / 2] & 0xffff0000u : v[0][j / 2] << 16);
}
// the sum over a row's 16 lanes up to the own one
template <int N>
__device__ __forceinline__ double cw_from_left(double v) {
  const uint64_t bits = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)bits, 0x110 + N, 0xf, 0xf, true);      // row_shr: zeros enter
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(bits >> 32), 0x110 + N, 0xf, 0xf, true);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ double cw_row_prefix(double v) {
  v += cw_from_left<1>(v);
  v += cw_from_left<2>(v);
  v += cw_from_left<4>(v);
  v += cw_from_left<8>(v);
  return v;
}

// exp of an exponent of 64 bits: what a float of it leaves out is small
__device__ __forceinline__ float cw_exp(double v) {
  const float hi = (float)v;
  const float e = expf(hi);
  return e + e * (float)(v - (double)hi);
}

template <int DT>
struct ChunkWalkLds {
  float sk[CW_RING][CW_TOKENS][16 * DT + 4], sq[CW_RING][CW_TOKENS][16 * DT + 4];
  float att[CW_RING][2][CW_TOKENS][CW_TOKENS + 4], low[2][2][CW_TOKENS][CW_TOKENS + 4], inv[2][CW_TOKENS][CW_TOKENS + 4];
  float pre[CW_RING][CW_TOKENS], post[CW_RING][CW_TOKENS], fac[CW_RING][CW_TOKENS];
  float unit_k[CW_RING][CW_TOKENS], unit_q[CW_RING][CW_TOKENS];
  double cum[CW_RING][CW_TOKENS];
};

template <typename T, int DT, bool DELTA, int OWNERS>       // states of up to 16 DT rows
__global__ __launch_bounds__((OWNERS + 5) * WAVE) void chunk_walk_kernel(
    const T* __restrict__ qkv, int64_t qkv_stride, int q_col, int k_col, int v_col, const float* __restrict__ gates,
    int64_t gate_stride, int a_col, int b_col, const float* __restrict__ dt_bias, const float* __restrict__ a_log,
    const float* __restrict__ d_skip, const int* __restrict__ seq_slot, const int* __restrict__ cu_rows,
    const int* __restrict__ q_len, float* __restrict__ state, float* __restrict__ out, int H, int G, int D, int P,
    float q_scale, float unit_eps, int write_state) {
  constexpr int N = CW_TOKENS, PER = 2 * DT;
  extern __shared__ __attribute__((aligned(16))) char cw_lds[];
  ChunkWalkLds<DT>& lds = *(ChunkWalkLds<DT>*)cw_lds;
  const int seq = blockIdx.x, head = blockIdx.y, group = head / (H / G);
  const int slot = seq_slot[seq], rows = q_len[seq];
  if (slot < 0 || rows <= 0) return;
  const int64_t first = cu_rows[seq];
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE, c = lane % 16, g = lane / 16;
  const int chunks = (rows + N - 1) / N;

  if (wave == OWNERS + 4) {                                  // ------------------------- decays and (I + L)^-1
    const float rate = expf(a_log[head]), bias = dt_bias[head];
    float gate_a[3], gate_b[3];
    auto fetch = [&](int n, float& a, float& b) __attribute__((always_inline)) {
      const float* gr = gates + (first + min(n * N + c, rows - 1)) * gate_stride + head;
      a = gr[a_col];
      b = DELTA ? gr[b_col] : 0.f;
    };
    auto decays = [&](int n, float a, float gb) __attribute__((always_inline)) {   // every 16 lanes a chunk's tokens
      const int b = n % CW_RING, left = rows - n * N;
      const float dt = cw_softplus(a + bias);
      double lg = -(double)rate * (double)dt;
      lg = lg < -1e6 ? -1e6 : lg;                            // nothing is left either way, and differences stay finite
      const double sum = cw_row_prefix(c < left ? lg : 0.0);
      const uint64_t bits = __builtin_bit_cast(uint64_t, sum);
      const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)bits, N - 1), hi = __builtin_amdgcn_readlane((int)(uint32_t)(bits >> 32), N - 1);
      const double all = __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
      if (lane < N) {
        lds.cum[b][lane] = sum;
        lds.pre[b][lane] = cw_exp(sum);
        lds.post[b][lane] = cw_exp(all - sum);
        lds.fac[b][lane] = c < left ? (DELTA ? 1.f / (1.f + expf(-gb)) : dt) : 0.f;
      }
    };
    // four lanes a column; each holds the values of every fourth row, a row's sum is one over the four
    auto invert = [&](int n) __attribute__((always_inline)) {
      const int col = lane / 4, sub = lane % 4;
      float x[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) x[k] = 0.f;
      vf4 l[2][N];                                           // columns sub, sub + 4, ... of every row, all asked for at once
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) l[h][i] = *(const vf4*)(lds.low[n & 1][h][i] + 4 * sub);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        float acc = 0.f;
#pragma unroll
        for (int k = 0; k < (i + 3) / 4; ++k) acc += (l[0][i][k] + l[1][i][k]) * x[k];
        const float v = (i == col ? 1.f : 0.f) - lanes_sum<4>(acc);
        x[i / 4] = sub == i % 4 ? v : x[i / 4];
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) lds.inv[n & 1][4 * k + sub][col] = x[k];
    };
#pragma unroll
    for (int m = 0; m < 3; ++m) fetch(m, gate_a[m], gate_b[m]);
#pragma unroll
    for (int m = 0; m < 3; ++m) decays(m, gate_a[m], gate_b[m]);
    fetch(3, gate_a[0], gate_b[0]);
    cw_barrier();
    cw_barrier();
    if (DELTA) invert(0);
    cw_barrier();
    for (int n = 0; n < chunks; ++n) {
      decays(n + 3, gate_a[0], gate_b[0]);                   // beyond the end: factors of no token
      fetch(n + 4, gate_a[0], gate_b[0]);
      if (DELTA) invert(n + 1);
      cw_barrier();
    }
    return;
  }

  if (wave >= OWNERS) {                                      // ------------------------------------------ helpers
    const int h = threadIdx.x - OWNERS * WAVE, tok = h >> 4, is_k = (h >> 3) & 1, part = h % 8, role = wave - OWNERS;
    vu4 x[3][PER / 8][2];
    auto fetch = [&](int n, vu4 (&to)[PER / 8][2]) __attribute__((always_inline)) {
      const T* src = qkv + (first + min(n * N + tok, rows - 1)) * qkv_stride + (is_k ? k_col : q_col) + group * D;
#pragma unroll
      for (int i = 0; i < PER / 8; ++i) cw_raw8(src + (part * PER + 8 * i < D ? part * PER + 8 * i : 0), to[i]);
    };
    auto stage = [&](int n, vu4 (&from)[PER / 8][2]) __attribute__((always_inline)) {
      const int b = n % CW_RING, left = rows - n * N;
      float v[PER];
#pragma unroll
      for (int i = 0; i < PER / 8; ++i) {
        const uint32_t keep = tok < left && part * PER + 8 * i < D ? ~0u : 0u;
#pragma unroll
        for (int w = 0; w < (int)sizeof(T) / 2; ++w) from[i][w] &= keep;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[8 * i + j] = cw_value<T>(from[i], j);
      }
      if (DELTA) {                                           // 1 / length: its power of two here, the rest later
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < PER; ++i) ss += v[i] * v[i];
        // rows beyond the end are zeros and stay so whatever unit_eps is: their factor is 1, not 1 / sqrt(0)
        const uint32_t bits = tok < left ? __float_as_uint(rsqrtf(lanes_sum<8>(ss) + unit_eps)) : __float_as_uint(1.f);
        const float power = __uint_as_float(bits & 0x7f800000u), rest = __uint_as_float((bits & 0x7fffffu) | 0x3f800000u);
#pragma unroll
        for (int i = 0; i < PER; ++i) v[i] *= power;
        if (part == 0) (is_k ? lds.unit_k : lds.unit_q)[b][tok] = is_k ? rest : rest * q_scale;
      }
      float* dst = (is_k ? lds.sk[b][tok] : lds.sq[b][tok]) + part * PER;
#pragma unroll
      for (int i = 0; i < PER; i += 4) *(vf4*)(dst + i) = vf4{v[i], v[i + 1], v[i + 2], v[i + 3]};
    };
    auto pairs = [&](int n) __attribute__((always_inline)) {
      const int b = n % CW_RING, half = role >> 1;
      if (!DELTA && (role & 1) == 0) return;
      const float* rows_a = (role & 1) ? lds.sq[b][c] : lds.sk[b][c];
      cw_f4 sum[4];
      sum[0] = sum[1] = sum[2] = sum[3] = cw_f4{0.f, 0.f, 0.f, 0.f};
      vf4 a[DT / 2], k[DT / 2];
#pragma unroll
      for (int u = 0; u < DT / 2; ++u) {
        const int t = half * (DT / 2) + u;
        a[u] = *(const vf4*)(rows_a + 16 * t + 4 * g);
        k[u] = *(const vf4*)(lds.sk[b][c] + 16 * t + 4 * g);
      }
      float m[4];
      const double at = lds.cum[b][c];
#pragma unroll
      for (int r = 0; r < 4; ++r) m[r] = cw_exp(lds.cum[b][4 * g + r] - at);
      vf4 f = {1.f, 1.f, 1.f, 1.f};                          // row i = 4 g + r, column j = c
      if (DELTA) f = *(const vf4*)(((role & 1) ? lds.unit_q[b] : lds.unit_k[b]) + 4 * g) * lds.unit_k[b][c];
      if (DELTA && (role & 1) == 0) f *= *(const vf4*)(lds.fac[b] + 4 * g);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < DT / 2; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[r] = cw_mfma(a[u][r], k[u][r], sum[r]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = 4 * g + r;
        const float v = ((sum[0][r] + sum[1][r]) + (sum[2][r] + sum[3][r])) * (f[r] * m[r]);
        if (role & 1) lds.att[b][half][i][c] = i >= c ? v : 0.f;
        else lds.low[n & 1][half][i][(c % 4) * 4 + c / 4] = i > c ? v : 0.f;
      }
    };
#pragma unroll
    for (int m = 0; m < 3; ++m) fetch(m, x[m]);
#pragma unroll
    for (int m = 0; m < 3; ++m) stage(m, x[m]);
    fetch(3, x[0]);
    cw_barrier();
    pairs(0);
    pairs(1);
    cw_barrier();
    cw_barrier();
    for (int n = 0; n < chunks; ++n) {                       // beyond the end: chunks of zeros
      stage(n + 3, x[0]);
      fetch(n + 4, x[0]);
      pairs(n + 2);
      cw_barrier();
    }
    return;
  }

  // -------------------------------------------------------------------------------------------------- owners
  __builtin_amdgcn_s_setprio(2);                             // the others' work is off the chain
  const int p = (blockIdx.z * OWNERS + wave) * 16 + c;
  const bool live = p < P;
  float* mine = state + (((int64_t)slot * H + head) * D) * P + p;
  cw_f4 S[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = 16 * t + 4 * g + r;
      S[t][r] = live && d < D ? mine[(int64_t)d * P] : 0.f;
    }
  const float skip = DELTA ? 0.f : d_skip[head];
  T next[4];
  const T* v_at = qkv + first * qkv_stride + v_col + head * P + (live ? p : 0);
  auto values = [&](int n) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 4; ++r) next[r] = v_at[min(n * N + 4 * g + r, rows - 1) * qkv_stride];
  };
  cw_f4 ks[4], qs[4];                                        // four sums each: short chains
  auto read_out = [&](int n) __attribute__((always_inline)) {
    const int b = n % CW_RING;
#pragma unroll
    for (int r = 0; r < 4; ++r) ks[r] = qs[r] = cw_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      vf4 k, q;
      if (DELTA) k = *(const vf4*)(lds.sk[b][c] + 16 * t + 4 * g);
      q = *(const vf4*)(lds.sq[b][c] + 16 * t + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (DELTA) ks[r] = cw_mfma(k[r], S[t][r], ks[r]);
        qs[r] = cw_mfma(q[r], S[t][r], qs[r]);
      }
    }
  };
  values(0);
  cw_barrier();
  cw_barrier();
  read_out(0);
  cw_barrier();
  for (int n = 0; n < chunks; ++n) {
    const int b = n % CW_RING, left = rows - n * N;
    const vf4 f = *(const vf4*)(lds.fac[b] + 4 * g);
    vf4 grown_k = *(const vf4*)(lds.pre[b] + 4 * g), grown_q = grown_k, to_end = *(const vf4*)(lds.post[b] + 4 * g);
    if (DELTA) {
      const vf4 uk = *(const vf4*)(lds.unit_k[b] + 4 * g);
      grown_k *= uk;
      grown_q *= *(const vf4*)(lds.unit_q[b] + 4 * g);
      to_end *= uk;
    }
    const float all = lds.pre[b][N - 1];
    cw_f4 u, o;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = live && 4 * g + r < left ? load_as_float(&next[r]) : 0.f;
      u[r] = f[r] * (DELTA ? v - grown_k[r] * ((ks[0][r] + ks[1][r]) + (ks[2][r] + ks[3][r])) : v);
      o[r] = grown_q[r] * ((qs[0][r] + qs[1][r]) + (qs[2][r] + qs[3][r])) + (DELTA ? 0.f : skip * v);
    }
    values(n + 1);                                           // beyond the end: the last row once more
    const cw_f4 rhs = u;
    if (DELTA) {
      const vf4 w = *(const vf4*)(lds.inv[n & 1][c] + 4 * g);
      u = cw_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < 4; ++r) u = cw_mfma(w[r], rhs[r], u);
    }
    const vf4 a = *(const vf4*)(lds.att[b][0][c] + 4 * g) + *(const vf4*)(lds.att[b][1][c] + 4 * g);
    const cw_f4 carried = o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o = cw_mfma(a[r], u[r], o);
    // A factor 0 keeps a token from those before it only while its u is a number. Where one is none (a bad row of the input),
    // its column is summed again over the tokens up to each one's own, as a walk row by row would.
    const uint64_t strays = __ballot(!(fabsf(u[0]) < INFINITY && fabsf(u[1]) < INFINITY && fabsf(u[2]) < INFINITY && fabsf(u[3]) < INFINITY));
    if (strays) {
      const bool again = (((strays >> c) | (strays >> (c + 16)) | (strays >> (c + 32)) | (strays >> (c + 48))) & 1) != 0;
      auto up_to_own = [&](const float (*one)[N + 4], const float (*two)[N + 4], cw_f4 x, cw_f4 sum) __attribute__((always_inline)) {
#pragma unroll 1
        for (int j4 = 0; j4 < N; j4 += 4)
#pragma unroll
          for (int jr = 0; jr < 4; ++jr) {
            const float xj = __shfl(x[jr], c + 4 * j4, WAVE);        // token j4 + jr of this column
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int i = 4 * g + r, j = j4 + jr;
              if (j <= i) sum[r] += (one[i][j] + (two != nullptr ? two[i][j] : 0.f)) * xj;
            }
          }
        return sum;
      };
      if (DELTA) {
        const cw_f4 own = up_to_own(lds.inv[n & 1], nullptr, rhs, cw_f4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int r = 0; r < 4; ++r) u[r] = again ? own[r] : u[r];
      }
      const cw_f4 own = up_to_own(lds.att[b][0], lds.att[b][1], u, carried);
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = again ? own[r] : o[r];
    }
    cw_f4 eu;
#pragma unroll
    for (int r = 0; r < 4; ++r) eu[r] = to_end[r] * u[r];
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      S[t] *= all;
#pragma unroll
      for (int r = 0; r < 4; ++r) S[t] = cw_mfma(lds.sk[b][4 * g + r][16 * t + c], eu[r], S[t]);
    }
    float* to = out + (first + n * N + 4 * g) * (int64_t)(H * P) + head * P + p;
    if (left >= N) {
      if (live) {
#pragma unroll
        for (int r = 0; r < 4; ++r) to[(int64_t)r * (H * P)] = o[r];
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (live && 4 * g + r < left) to[(int64_t)r * (H * P)] = o[r];
    }
    read_out(n + 1);                                         // beyond the end: of zeros, and not used
    cw_barrier();
  }
  if (!write_state || !live) return;
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = 16 * t + 4 * g + r;
      if (d < D) mine[(int64_t)d * P] = S[t][r];
    }
}

// What the kernel takes: whole pieces of 8 values of q and k at 16-byte addresses, states of at most 128 rows.
static bool chunk_walk_takes(const void* qkv, int64_t stride, int q_col, int k_col, int D) {
  return D % 8 == 0 && D <= 128 && q_col % 8 == 0 && k_col % 8 == 0 && stride % 8 == 0 && ((uintptr_t)qkv & 15) == 0;
}

template <bool DELTA>
static int chunk_walk_run(const void* qkv, int64_t stride, int q_col, int k_col, int v_col, const float* gates, int64_t gate_stride,
                          int a_col, int b_col, const float* dt_bias, const float* a_log, const float* d_skip, const int* seq_slot,
                          const int* cu_rows, const int* q_len, float* state, float* out, int n_seqs, int H, int G, int D, int P,
                          float q_scale, float unit_eps, int write_state, int is_f32, hipStream_t stream) {
  // 32 columns a workgroup while that fills the chip at most once: 16 heads of 128 x 128, 5,099 rows of four sequences 385
  // us against 429 with 64 (measured with two barriers a chunk); more workgroups than compute units would wait for a turn
  const bool narrow = (int64_t)n_seqs * H * ((P + 31) / 32) <= 256;
#define CW_LAUNCH(TT, DT, OW)                                                                                              \
  do {                                                                                                                     \
    if (sizeof(ChunkWalkLds<DT>) > 64 * 1024 &&                                                                            \
        hipFuncSetAttribute((const void*)chunk_walk_kernel<TT, DT, DELTA, OW>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                            (int)sizeof(ChunkWalkLds<DT>)) != hipSuccess)                                                  \
      return -1;                                                                                                           \
    hipLaunchKernelGGL((chunk_walk_kernel<TT, DT, DELTA, OW>), dim3(n_seqs, H, (P + 16 * OW - 1) / (16 * OW)),             \
                       dim3((OW + 5) * WAVE), sizeof(ChunkWalkLds<DT>), stream, (const TT*)qkv, stride, q_col, k_col,      \
                       v_col, gates, gate_stride, a_col, b_col, dt_bias, a_log, d_skip, seq_slot, cu_rows, q_len, state,   \
                       out, H, G, D, P, q_scale, unit_eps, write_state);                                                   \
  } while (0)
#define CW_PICK(TT)                                                                                                        \
  do {                                                                                                                     \
    if (D <= 64) { if (narrow) CW_LAUNCH(TT, 4, 2); else CW_LAUNCH(TT, 4, 4); }                                            \
    else { if (narrow) CW_LAUNCH(TT, 8, 2); else CW_LAUNCH(TT, 8, 4); }                                                    \
  } while (0)
  if (is_f32) CW_PICK(float); else CW_PICK(bf16_t);
#undef CW_PICK
#undef CW_LAUNCH
  return DRYFT_LAUNCH_CHECK();
}
