// Causal grouped-query attention over the paged cache for the float32 path, on the matrix cores' full-precision
// instruction (v_mfma_f32_16x16x4_f32), keys and values of one width, a multiple of 16 up to 256:
//
//   s[j] = (q . k[j]) * scale  for  lo <= j <= pos,   p = softmax(s),   o = sum_j p[j] v[j]
//
// (reference: engine/dryft_qwen3/model.py:172-177, 254-257), lo = 0 or pos - window + 1; query head h reads kv head
// h / group. A workgroup takes 16 query columns of one kv head: the heads of one row's group (decoding: a workgroup per row,
// kv head and 16 heads of its group), or 16 rows of a sequence for one head (prompts: a workgroup per tile of 16 rows and
// head). Its waves take half pages (32 keys) in turn, each with a running maximum and sum of its own, and meet in LDS.
//
// Scores of 16 keys are C[key, column] = K . q^T: lane (c, g) holds keys 4g .. 4g + 3 of column c, which is what the second
// product, O^T[feature, column] += V^T . P, takes as its operand, one entry an instruction; a page of values keeps the
// positions of a half page in the order that gives a lane its eight of both tiles of 16 keys as 32 contiguous bytes
// (value_column). So scores never leave registers, and every line of a page is read once by one wave for all columns, where
// the kernel of one workgroup a (row, head) (attn_rows.hip) read every key with 16 bytes a line and request, once per head
// of the group. Between launches that stream other memory, us, against that kernel: Qwen3-0.6B's heads, one sequence, one row at
// 20 / 280 / 1,024 keys 6.9 / 15.8 / 39 (8.1 / 20.5 / 51), four sequences of 150 prompt rows 35 (115); in a traced serving pass
// decoding at 10 to 280 keys 14.6, 525 prompt rows 36.8.
// In decoding a compute unit takes in 35 KB/us, a half page of 128 features is 32 KB, and few rows leave most units without work: then
// a row's keys go over several workgroups (SPLIT) of fewer waves (by what a unit takes in at once: 2, 4 or 8), whose last one adds up
// their partial results. 16 heads on 8 of 128, one workgroup a row and kv head / split, us: one sequence of 280 / 1,024 / 4,096 keys 15.1
// / 37.0 / 126 and 10.6 / 11.5 / 17.9, four 15.3 / 39 / 135 and 10.9 / 14.2 / 35, four of 20 / 150 6.1 / 10.6 and 6.2 / 10.7; 8 on 1 of
// 64, four of 150 / 1,024 7.8 / 22.2 and 7.2 / 10.3. Which steps take which form, and where the other kernel stays ahead:
// `float32_form` and `float32_splits` in parts/attention.py.
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;

struct AttnF32 {
  const float* q;                 // [rows, n_heads, D]
  float* k_pages;                 // written where the row's own key and value are appended
  float* v_pages;
  const int* page_table;
  int max_pages;
  const int* row_slot;            // decoding
  const int* row_pos;
  const int* seq_slot;            // prompts
  const int* cu_rows;
  const int* tile_cu;
  const int* seq_start;
  int n_seqs;
  float* out;                     // [rows, n_heads, D]
  int n_heads, n_kv, head_dim;
  float scale;
  int window;
  int n_splits;                   // splits of a decoding row's keys, their partial results, and counters that are zeros between launches
  float* part_o;                  // [rows, n_heads, n_splits, D]
  float* part_ml;                 // [rows, n_heads, n_splits, 2]
  int* arrivals;                  // [rows, kv heads * blocks of 16 heads]
  // decoding with the work of the norm / rotation / append kernel: a row's q heads | k heads | v heads as the projection left them
  const float* qkv;
  int64_t stride;
  const float *q_w, *k_w;         // per-head norms, or null
  float eps;
  const float *cos_t, *sin_t;     // [positions, head_dim / 2]
  int write_kv;
};

// Values that workgroups of one launch hand to one another: past the caches that the chip's compute dies keep for themselves.
__device__ __forceinline__ void store_far(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float load_far(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

#define F32_SPLIT_WAVES(DT) ((DT) <= 4 ? 8 : (DT) <= 8 ? 4 : 2)
#define F32_MAX_SPLITS 32

template <int DT, int WAVES, bool TILES, bool SPLIT = false, bool FUSED = false>
__global__ __launch_bounds__(WAVES * WAVE) void attn_f32_kernel(AttnF32 a) {
  extern __shared__ __align__(16) float attn_f32_lds[];
  constexpr int D = 16 * DT, OS = D + 1;
  float* merge_o = attn_f32_lds;                           // [WAVES][16][OS]
  float* merge_m = merge_o + WAVES * 16 * OS;              // [WAVES][16]
  float* merge_l = merge_m + WAVES * 16;
  const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE, c = lane % 16, g = lane / 16;
  const int group = a.n_heads / a.n_kv;
  int slot, kvh, columns, pos, first_pos, last_pos;        // pos: this lane's column's; of the first and the last column
  int64_t q_at;                                            // this lane's column of q and out
  if (TILES) {
    const int tile = blockIdx.x, head = blockIdx.y;
    if (tile >= a.tile_cu[a.n_seqs]) return;
    int lo = 0, hi = a.n_seqs - 1;                         // the sequence whose tiles hold this one
    while (lo < hi) {
      const int mid = (lo + hi + 1) / 2;
      if (a.tile_cu[mid] <= tile) lo = mid;
      else hi = mid - 1;
    }
    const int r0 = 16 * (tile - a.tile_cu[lo]);
    slot = a.seq_slot[lo];
    kvh = head / group;
    columns = min(16, a.cu_rows[lo + 1] - a.cu_rows[lo] - r0);
    first_pos = a.seq_start[lo] + r0;
    last_pos = first_pos + columns - 1;
    pos = first_pos + min(c, columns - 1);
    q_at = ((int64_t)(a.cu_rows[lo] + r0 + min(c, columns - 1)) * a.n_heads + head) * D;
  } else {
    const int blocks = (group + 15) / 16;
    const int64_t row = blockIdx.x;
    kvh = blockIdx.y / blocks;
    const int h0 = (blockIdx.y % blocks) * 16;
    slot = a.row_slot[row];
    columns = min(16, group - h0);
    first_pos = last_pos = pos = a.row_pos[row];
    q_at = (row * a.n_heads + kvh * group + h0 + min(c, columns - 1)) * D;
    if (slot < 0 && SPLIT && blockIdx.z > 0) return;
    if (slot < 0) {                                        // a row that sits out: zeros
      const int64_t at = (row * a.n_heads + kvh * group + h0) * D;
      for (int i = threadIdx.x; i < columns * D; i += blockDim.x) a.out[at + i] = 0.f;
      return;
    }
  }
  if (slot < 0) return;                                    // no tile belongs to a sequence that sits out
  const int lo_col = a.window > 0 ? max(0, pos - a.window + 1) : 0;
  const int lo_all = a.window > 0 ? max(0, first_pos - a.window + 1) : 0;
  const int* table = a.page_table + (int64_t)slot * a.max_pages;
  // half pages in turn over the waves of all splits; a split whose first wave has none has nothing to say
  const int stride = SPLIT ? WAVES * a.n_splits : WAVES, first_unit = lo_all / 32 + (SPLIT ? WAVES * blockIdx.z : 0);
  if (SPLIT && 32 * first_unit > last_pos) return;
  const int live = SPLIT ? min(a.n_splits, (last_pos / 32 - lo_all / 32 + WAVES) / WAVES) : 1;
  f32x4 qv[DT];
  f32x4 own_k[FUSED ? DT : 1];                             // the row's own key, as the lanes of its column hold it, and value
  float own_v[FUSED ? DT : 1];
  const bool owner = FUSED && a.write_kv && last_pos / 32 >= first_unit + wave && (last_pos / 32 - first_unit - wave) % stride == 0;
  if constexpr (FUSED) {
    // Heads are normed and turned as they lie: a lane's features 16 t + 4g .. + 3 turn with those of t + DT / 2. The wave that reads the
    // half page of the row's own position also makes the new key and value, puts them into its operands and appends them.
    const float* src = a.qkv + (int64_t)blockIdx.x * a.stride;
    const float* qp = src + (int64_t)(kvh * group + min(c, columns - 1)) * D + 4 * g;
    f32x4 wq[DT], wk[DT], cs[DT / 2], sn[DT / 2];
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      qv[t] = *(const f32x4*)(qp + 16 * t);
      if (a.q_w != nullptr) wq[t] = *(const f32x4*)(a.q_w + 16 * t + 4 * g);
    }
#pragma unroll
    for (int t = 0; t < DT / 2; ++t) {
      cs[t] = *(const f32x4*)(a.cos_t + (int64_t)pos * (D / 2) + 16 * t + 4 * g);
      sn[t] = *(const f32x4*)(a.sin_t + (int64_t)pos * (D / 2) + 16 * t + 4 * g);
    }
    if (owner) {
      const float* kq = src + (int64_t)(a.n_heads + kvh) * D + 4 * g;
      const float* vq = src + (int64_t)(a.n_heads + a.n_kv + kvh) * D + c;
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        own_k[t] = *(const f32x4*)(kq + 16 * t);
        own_v[t] = vq[16 * t];
        if (a.k_w != nullptr) wk[t] = *(const f32x4*)(a.k_w + 16 * t + 4 * g);
      }
    }
    auto turn = [&](f32x4 (&x)[DT], const f32x4 (&w)[DT], bool normed) {
      if (normed) {
        float ss = 0.f;
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) ss += x[t][i] * x[t][i];
        ss += __shfl_xor(ss, 16, WAVE);
        ss += __shfl_xor(ss, 32, WAVE);
        const float inv = rsqrtf(ss / (float)D + a.eps);
#pragma unroll
        for (int t = 0; t < DT; ++t) x[t] = x[t] * inv * w[t];
      }
#pragma unroll
      for (int t = 0; t < DT / 2; ++t) {
        const f32x4 one = x[t], two = x[t + DT / 2];
        x[t] = one * cs[t] - two * sn[t];
        x[t + DT / 2] = two * cs[t] + one * sn[t];
      }
    };
    turn(qv, wq, a.q_w != nullptr);
    if (owner) turn(own_k, wk, a.k_w != nullptr);
  } else {
#pragma unroll
    for (int t = 0; t < DT; ++t) qv[t] = *(const f32x4*)(a.q + q_at + 16 * t + 4 * g);
  }
  f32x4 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;                            // l: over the keys of this lane alone
  constexpr bool V_EARLY = DT <= 8;                        // wider heads have no registers for the values that soon
  int u = first_unit + wave;
  int page = 32 * u <= last_pos ? table[u / 2] : -1;
  for (; 32 * u <= last_pos; u += stride) {
    const int here = page;
    page = 32 * (u + stride) <= last_pos ? table[(u + stride) / 2] : -1;
    if (here < 0) continue;
    const int64_t base = ((int64_t)here * a.n_kv + kvh) * PAGE_TOKENS * D;
    const float* kp = a.k_pages + base + (int64_t)(32 * (u & 1) + c) * D + 4 * g;
    const float* vp = a.v_pages + base + (int64_t)c * PAGE_TOKENS + 32 * (u & 1) + 8 * g;
    // everything the half page needs is asked for at once: one trip to memory, not one for the keys and one for the values
    f32x4 kv[2][DT], vv[DT][2];
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int t = 0; t < DT; ++t) kv[half][t] = *(const f32x4*)(kp + 16 * half * D + 16 * t);
    if (V_EARLY) {
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int half = 0; half < 2; ++half) vv[t][half] = *(const f32x4*)(vp + (int64_t)16 * t * PAGE_TOKENS + 4 * half);
    }
    if constexpr (FUSED) {
      static_assert(V_EARLY, "the own value goes into what has been asked for");
      if (owner && u == last_pos / 32) {
        const int in_page = last_pos % PAGE_TOKENS, place = value_column(in_page) % 32;
#pragma unroll
        for (int t = 0; t < DT; ++t) {
#pragma unroll
          for (int half = 0; half < 2; ++half) {
            if (c == in_page % 16 && half == in_page % 32 / 16) kv[half][t] = own_k[t];
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (g == place / 8 && 4 * half + i == place % 8) vv[t][half][i] = own_v[t];
          }
          if (c == 0) *(f32x4*)(a.k_pages + base + (int64_t)in_page * D + 16 * t + 4 * g) = own_k[t];
          if (g == 0) a.v_pages[base + (int64_t)(16 * t + c) * PAGE_TOKENS + value_column(in_page)] = own_v[t];
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // four sums side by side: an instruction need not wait for the one before it
    f32x4 s[2], odd[2];
#pragma unroll
    for (int half = 0; half < 2; ++half) s[half] = odd[half] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int i = 0; i < 4; i += 2)
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          s[half] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[half][t][i], qv[t][i], s[half], 0, 0, 0);
          odd[half] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[half][t][i + 1], qv[t][i + 1], odd[half], 0, 0, 0);
        }
#pragma unroll
    for (int half = 0; half < 2; ++half) s[half] += odd[half];
    float top = -INFINITY;
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = 32 * u + 16 * half + 4 * g + i;
        s[half][i] = j >= lo_col && j <= pos ? s[half][i] * a.scale : -INFINITY;
        top = fmaxf(top, s[half][i]);
      }
    top = fmaxf(top, __shfl_xor(top, 16, WAVE));
    top = fmaxf(top, __shfl_xor(top, 32, WAVE));
    const float m_new = fmaxf(m, top);
    // a column that has seen no key yet has m_new = -inf: its weights are zeros
    const float keep = m_new == -INFINITY ? 0.f : expf(m - m_new);
    f32x4 p[2];
    float added = 0.f;
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[half][i] = s[half][i] == -INFINITY ? 0.f : expf(s[half][i] - m_new);
        added += p[half][i];
      }
    l = l * keep + added;
    m = m_new;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      o[t] *= keep;
      if (!V_EARLY) {
#pragma unroll
        for (int half = 0; half < 2; ++half) vv[t][half] = *(const f32x4*)(vp + (int64_t)16 * t * PAGE_TOKENS + 4 * half);
      }
    }
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < DT; ++t) o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[t][half][i], p[half][i], o[t], 0, 0, 0);
  }
  l += __shfl_xor(l, 16, WAVE);
  l += __shfl_xor(l, 32, WAVE);
  // o[t][i] is feature 16 t + 4g + i of column c
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) merge_o[(wave * 16 + c) * OS + 16 * t + 4 * g + i] = o[t][i];
  if (g == 0) {
    merge_m[wave * 16 + c] = m;
    merge_l[wave * 16 + c] = l;
  }
  __syncthreads();
  const int64_t out_step = TILES ? (int64_t)a.n_heads * D : D;           // from one column to the next
  const int64_t out_at = q_at - (int64_t)min(c, columns - 1) * out_step;  // of the first
  for (int idx = threadIdx.x; idx < columns * D; idx += blockDim.x) {
    const int col = idx / D, d = idx % D;
    float top = -INFINITY;
#pragma unroll
    for (int v = 0; v < WAVES; ++v) top = fmaxf(top, merge_m[v * 16 + col]);
    float sum = 0.f, total = 0.f;
#pragma unroll
    for (int v = 0; v < WAVES; ++v) {
      const float mv = merge_m[v * 16 + col];
      const float wgt = mv == -INFINITY ? 0.f : expf(mv - top);
      total += wgt * merge_l[v * 16 + col];
      sum += wgt * merge_o[(v * 16 + col) * OS + d];
    }
    if (SPLIT && live > 1) {
      const int64_t at = (out_at / D + col) * a.n_splits + blockIdx.z;
      store_far(a.part_o + at * D + d, sum);
      if (d == 0) {
        store_far(a.part_ml + 2 * at, top);
        store_far(a.part_ml + 2 * at + 1, total);
      }
      continue;
    }
    // whatever the total is: a score of NaN or +inf, or none but -inf (0 / 0), leaves no number, as in the softmax
    a.out[out_at + col * out_step + d] = sum / total;
  }
  if (!SPLIT || live == 1) return;
  // The workgroup that comes last of a row's splits adds them up, in their order, so that results do not depend on timing. Nobody
  // waits: the others are gone by then. What they wrote is counted only once it has arrived.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __shared__ int came_last;
  __syncthreads();
  if (threadIdx.x == 0) {
    int* count = a.arrivals + (int64_t)blockIdx.x * gridDim.y + blockIdx.y;
    const int before = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    came_last = before == live - 1;
    if (came_last) __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // for the next launch
  }
  __syncthreads();
  if (!came_last) return;
  auto ask = [&](float (&o8)[8], int idx, int v0) {        // eight partial results on their way at a time
    const float* po = a.part_o + (out_at / D + idx / D) * a.n_splits * D + idx % D;
#pragma unroll
    for (int v = 0; v < 8; ++v)
      if (v0 + v < live) o8[v] = load_far(po + (int64_t)(v0 + v) * D);
  };
  float o8[8];
  if (threadIdx.x < columns * D) ask(o8, threadIdx.x, 0);  // the first of them along with the weights
  float* ml = attn_f32_lds;                                // [16][F32_MAX_SPLITS][2], where the waves' results were
  for (int i = threadIdx.x; i < columns * live; i += blockDim.x) {
    const int64_t at = (out_at / D + i / live) * a.n_splits + i % live;
    ml[2 * (i / live * F32_MAX_SPLITS + i % live)] = load_far(a.part_ml + 2 * at);
    ml[2 * (i / live * F32_MAX_SPLITS + i % live) + 1] = load_far(a.part_ml + 2 * at + 1);
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < columns * D; idx += blockDim.x) {
    const int col = idx / D, d = idx % D;
    const float* mine = ml + 2 * F32_MAX_SPLITS * col;
    float top = -INFINITY;
    for (int v = 0; v < live; ++v) top = fmaxf(top, mine[2 * v]);
    float sum = 0.f, total = 0.f;
    for (int v0 = 0; v0 < live; v0 += 8) {
      if (v0 > 0 || idx != (int)threadIdx.x) ask(o8, idx, v0);
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        if (v0 + v >= live) continue;
        const float mv = mine[2 * (v0 + v)], wgt = mv == -INFINITY ? 0.f : expf(mv - top);
        total += wgt * mine[2 * (v0 + v) + 1];
        sum += wgt * o8[v];
      }
    }
    a.out[out_at + col * out_step + d] = sum / total;
  }
}

template <int DT, int WAVES, bool TILES, bool SPLIT = false, bool FUSED = false>
static int launch_attn_f32(const AttnF32& a, dim3 grid, hipStream_t stream) {
  constexpr int merge = WAVES * 16 * (16 * DT + 1 + 2) * 4, weights = SPLIT ? 16 * F32_MAX_SPLITS * 2 * 4 : 0;
  constexpr int lds = merge > weights ? merge : weights;
  static_assert(lds <= 160 * 1024, "the merge must fit a compute unit's LDS");
  auto kernel = attn_f32_kernel<DT, WAVES, TILES, SPLIT, FUSED>;
  static bool raised = false;                              // more dynamic LDS than the default limit allows
  if (lds > 64 * 1024 && !raised) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess) return -2;
    raised = true;
  }
  hipLaunchKernelGGL(kernel, grid, dim3(WAVES * WAVE), lds, stream, a);
  return DRYFT_LAUNCH_CHECK();
}

template <bool TILES>
static int dispatch_attn_f32(const AttnF32& a, dim3 grid, hipStream_t stream) {
  if (a.n_kv <= 0 || a.n_heads % a.n_kv || a.head_dim <= 0 || a.head_dim % 16 || a.head_dim > 256 || grid.y > 65535 ||
      (((uintptr_t)a.q | (uintptr_t)a.k_pages | (uintptr_t)a.v_pages) & 15))
    return -1;
#define ATTN_F32(DTV, WV)                                                                                      \
  case DTV:                                                                                                      \
    if (!TILES && a.n_splits > 1) return launch_attn_f32<DTV, F32_SPLIT_WAVES(DTV), false, true>(a, grid, stream);    \
    return launch_attn_f32<DTV, WV, TILES>(a, grid, stream)
  switch (a.head_dim / 16) {                               // eight waves where the merge of a decoding row fits twice a unit
    ATTN_F32(1, 4); ATTN_F32(2, 4); ATTN_F32(3, 4); ATTN_F32(4, 4);
    ATTN_F32(5, 4); ATTN_F32(6, 4); ATTN_F32(7, 4); ATTN_F32(8, (TILES ? 4 : 8));
    ATTN_F32(9, 4); ATTN_F32(10, 4); ATTN_F32(11, 4); ATTN_F32(12, 4);
    ATTN_F32(13, 4); ATTN_F32(14, 4); ATTN_F32(15, 4); ATTN_F32(16, 4);
  }
#undef ATTN_F32
  return -1;
}

// One row per sequence with the work of dryft_qk_norm_rope_kv: heads of 32, 64, 96 or (split) 128 features that turn as a whole, at most
// 16 query heads a kv head. Splits and their scratch as below. Two launches / one, us: 16 heads on 8 of 128, four sequences of 150 / 1,024
// keys 14.6 / 11.7 and 18.8 / 16.1; 8 on 1 of 64 10.2 / 8.8 and 13.6 / 12.5; 64 sequences of 150, 12 heads of 96, 38.5 / 34.1. -2: sizes or addresses that the kernel does not take.
DRYFT_API int dryft_attn_f32_fused(const void* qkv, int64_t stride, const float* q_w, const float* k_w, float eps, const float* cos_t,
                                   const float* sin_t, int write_kv, void* k_pages, void* v_pages, const int* page_table,
                                   int max_pages, const int* row_slot, const int* row_pos, void* out, int n_rows, int n_heads,
                                   int n_kv, int head_dim, float scale, int window, int n_splits, float* part_o, float* part_ml,
                                   int* arrivals, hipStream_t stream) {
  if (n_rows <= 0) return 0;
  if (n_kv <= 0 || n_heads % n_kv || n_splits < 1 || n_splits > F32_MAX_SPLITS || (n_splits > 1 && !(part_o && part_ml && arrivals)))
    return -1;
  if (head_dim <= 0 || head_dim % 32 || head_dim > 128 || n_heads > 16 * n_kv || n_kv > 65535 || stride % 4 || !cos_t || !sin_t ||
      (q_w == nullptr) != (k_w == nullptr) ||
      (((uintptr_t)qkv | (uintptr_t)q_w | (uintptr_t)k_w | (uintptr_t)cos_t | (uintptr_t)sin_t | (uintptr_t)k_pages | (uintptr_t)v_pages) & 15))
    return -2;
  AttnF32 a = {nullptr, (float*)k_pages, (float*)v_pages, page_table, max_pages, row_slot, row_pos, nullptr, nullptr, nullptr, nullptr, 0,
               (float*)out, n_heads, n_kv, head_dim, scale, window, n_splits, part_o, part_ml, arrivals, (const float*)qkv, stride, q_w,
               k_w, eps, cos_t, sin_t, write_kv};
  const dim3 grid(n_rows, n_kv, n_splits);
  if (n_splits > 1) {
    switch (head_dim / 16) {
      case 2: return launch_attn_f32<2, F32_SPLIT_WAVES(2), false, true, true>(a, grid, stream);
      case 4: return launch_attn_f32<4, F32_SPLIT_WAVES(4), false, true, true>(a, grid, stream);
      case 6: return launch_attn_f32<6, F32_SPLIT_WAVES(6), false, true, true>(a, grid, stream);
      case 8: return launch_attn_f32<8, F32_SPLIT_WAVES(8), false, true, true>(a, grid, stream);
    }
  }
  switch (head_dim / 16) {
    case 2: return launch_attn_f32<2, 4, false, false, true>(a, grid, stream);
    case 4: return launch_attn_f32<4, 4, false, false, true>(a, grid, stream);
    case 6: return launch_attn_f32<6, 4, false, false, true>(a, grid, stream);
  }
  return -2;                                               // 128 features in eight waves: no registers for the new key
}

// One row per sequence or any rows: each on its own, by its slot and position. With n_splits > 1 a row's keys go over so many
// workgroups (partial results and counters as in AttnF32).
DRYFT_API int dryft_attn_f32_rows(const void* q, const void* k_pages, const void* v_pages, const int* page_table,
                                  int max_pages, const int* row_slot, const int* row_pos, void* out, int n_rows, int n_heads,
                                  int n_kv, int head_dim, float scale, int window, int n_splits, float* part_o, float* part_ml,
                                  int* arrivals, hipStream_t stream) {
  if (n_rows <= 0) return 0;
  if (n_kv <= 0 || n_splits < 1 || n_splits > F32_MAX_SPLITS || (n_splits > 1 && !(part_o && part_ml && arrivals))) return -1;
  AttnF32 a = {(const float*)q, (float*)k_pages, (float*)v_pages, page_table, max_pages, row_slot, row_pos,
               nullptr, nullptr, nullptr, nullptr, 0, (float*)out, n_heads, n_kv, head_dim, scale, window, n_splits, part_o, part_ml,
               arrivals};
  const int blocks = (n_heads / n_kv + 15) / 16;
  return dispatch_attn_f32<false>(a, dim3(n_rows, n_kv * blocks, n_splits), stream);
}

// Rows in tiles of 16 of one sequence (tile_cu: their prefix sums over the sequences; max_tiles bounds their number).
// Rows of sequences that sit out are not visited.
DRYFT_API int dryft_attn_f32_tiles(const void* q, const void* k_pages, const void* v_pages, const int* page_table,
                                   int max_pages, const int* seq_slot, const int* cu_rows, const int* tile_cu,
                                   const int* seq_start, int n_seqs, int max_tiles, void* out, int n_heads, int n_kv,
                                   int head_dim, float scale, int window, hipStream_t stream) {
  if (n_seqs <= 0 || max_tiles <= 0) return 0;
  AttnF32 a = {(const float*)q, (float*)k_pages, (float*)v_pages, page_table, max_pages, nullptr, nullptr,
               seq_slot, cu_rows, tile_cu, seq_start, n_seqs, (float*)out, n_heads, n_kv, head_dim, scale, window, 1, nullptr, nullptr, nullptr};
  return dispatch_attn_f32<true>(a, dim3(max_tiles, n_heads), stream);
}
