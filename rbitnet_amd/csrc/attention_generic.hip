// Causal attention of each token over its sequence's paged cache: any head_dim up to
// 512, any number of heads and groups, float32 or bfloat16 storage, float32 arithmetic
// throughout (scores, softmax, weighted sum).  Float32 heads of up to 128 numbers run on the
// matrix cores (the last kernel); the others take one workgroup per
// (token, query head): one wave when the step has many tokens, up to 8 waves that share the pages of the context and merge
// their running softmax states through LDS when it has few (a decode step of 8 sequences and
// 32 heads would otherwise leave three quarters of the GPU idle, each wave walking its whole
// context alone).
//
// Reference: kv head = q head / (Hq / Hk); s[p] = (q . K[p]) * scale for p <= pos;
// softmax with the maximum subtracted; out = sum_p s[p] V[p]  (llama/model.rs:260-289,
// softmax :102-114).  The softmax is computed page by page with a running maximum, which
// is the same value up to rounding.
#include <math.h>

#include "api.h"
#include "common.h"
#include "mfma.h"

#define AG_MAX_D 512
#define AG_MAX_D_VEC 256      // the 16-byte kernel deals a row's quads to the lanes of one wave

#define AG_MAX_WAVES 8

template <typename T>
__global__ __launch_bounds__(RB_WAVE * AG_MAX_WAVES) void attention_generic_kernel(
    const T* __restrict__ q, const T* __restrict__ k_pages, const T* __restrict__ v_pages, T* __restrict__ out,
    const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ tok_seq,
    const int32_t* __restrict__ block_table, int bt_stride, int n_heads, int n_kv, int head_dim, float scale,
    int window, const float* __restrict__ sinks, int keep_first, float softcap, int chunk, const float* __restrict__ sig_bias) {
  __shared__ float qs[AG_MAX_D];
  __shared__ float ps_all[AG_MAX_WAVES][RB_PAGE];
  __shared__ float red_m[AG_MAX_WAVES], red_l[AG_MAX_WAVES];
  __shared__ float red_acc[AG_MAX_WAVES][AG_MAX_D];
  const int t = blockIdx.x;
  const int h = blockIdx.y;
  const int lane = threadIdx.x & (RB_WAVE - 1);
  const int wave = threadIdx.x / RB_WAVE, n_waves = blockDim.x / RB_WAVE;
  float* ps = ps_all[wave];
  const int pos = tok_pos[t];
  const int kvh = h / (n_heads / n_kv);
  const int lo = first_visible(pos, window, chunk);
  const int32_t* pages = block_table + (size_t)tok_seq[t] * bt_stride;

  const T* qrow = q + ((size_t)t * n_heads + h) * head_dim;
  for (int d = threadIdx.x; d < head_dim; d += blockDim.x) qs[d] = Num<T>::load(qrow + d);
  __syncthreads();

  // sigmoid weights (sig_bias): a key's weight is sigmoid(score + sig_bias[h]) by itself, so the maximum stays 0, nothing is
  // rescaled and nothing divided
  const float sb = sig_bias ? sig_bias[h] : 0.f;
  float m_run = sig_bias ? 0.f : -INFINITY, l_run = 0.f;
  float acc[AG_MAX_D / RB_WAVE];
#pragma unroll
  for (int i = 0; i < AG_MAX_D / RB_WAVE; ++i) acc[i] = 0.f;

  // the pages that hold visible keys: those of the kept first tokens that lie before the window's first page, then the
  // window's (every one of them holds at least one visible key)
  const int lo_page = lo / RB_PAGE;
  const int kept_pages = keep_first > 0 ? (keep_first + RB_PAGE - 1) / RB_PAGE : 0;
  const int n_first = kept_pages < lo_page ? kept_pages : lo_page;
  const int n_walk = n_first + pos / RB_PAGE - lo_page + 1;
  for (int walk = wave; walk < n_walk; walk += n_waves) {
    const int pg = walk < n_first ? walk : lo_page + walk - n_first;
    const size_t base = ((size_t)pages[pg] * n_kv + kvh) * RB_PAGE * head_dim;
    const int p = pg * RB_PAGE + lane;
    float s = -INFINITY;
    if (p <= pos && (p >= lo || p < keep_first)) {
      const T* krow = k_pages + base + (size_t)lane * head_dim;
      float dot = 0.f;
      for (int d = 0; d < head_dim; ++d) dot = fmaf(qs[d], Num<T>::load(krow + d), dot);
      s = dot * scale;
      if (softcap > 0.f) s = softcap * tanhf(s / softcap);
    }
    const float m_new = sig_bias ? 0.f : fmaxf(m_run, wave_max(s));      // finite: the page holds at least one valid key
    const float pexp = (s == -INFINITY) ? 0.f : (sig_bias ? 1.0f / (1.0f + expf(-(s + sb))) : expf(s - m_new));
    const float corr = (m_run == -INFINITY) ? 0.f : expf(m_run - m_new);
    l_run = l_run * corr + wave_sum(pexp);
    m_run = m_new;
    // ps belongs to this wave alone; a wave's LDS accesses complete in order
    ps[lane] = pexp;
    __builtin_amdgcn_wave_barrier();
    const int j_lo = (pg * RB_PAGE < lo && pg * RB_PAGE >= keep_first) ? lo - pg * RB_PAGE : 0;      // keys between carry weight 0
    const int j_hi = (pg * RB_PAGE + RB_PAGE - 1 > pos) ? pos - pg * RB_PAGE : RB_PAGE - 1;
#pragma unroll
    for (int i = 0; i < AG_MAX_D / RB_WAVE; ++i) {
      const int d = lane + i * RB_WAVE;
      if (d < head_dim) {
        float a = acc[i] * corr;
        const T* vcol = v_pages + base + d;
        for (int j = j_lo; j <= j_hi; ++j) a = fmaf(ps[j], Num<T>::load(vcol + (size_t)j * head_dim), a);
        acc[i] = a;
      }
    }
  }
  // ---- the waves' states into one (a wave without pages holds m = -inf, l = 0, acc = 0)
  if (n_waves > 1) {
    if (lane == 0) {
      red_m[wave] = m_run;
      red_l[wave] = l_run;
    }
#pragma unroll
    for (int i = 0; i < AG_MAX_D / RB_WAVE; ++i) {
      const int d = lane + i * RB_WAVE;
      if (d < head_dim) red_acc[wave][d] = acc[i];
    }
    __syncthreads();
    if (wave != 0) return;
    float mx = red_m[0];
    for (int w = 1; w < n_waves; ++w) mx = fmaxf(mx, red_m[w]);
    m_run = mx;
    l_run = 0.f;
#pragma unroll
    for (int i = 0; i < AG_MAX_D / RB_WAVE; ++i) acc[i] = 0.f;
    for (int w = 0; w < n_waves; ++w) {
      const float f = (red_m[w] == -INFINITY) ? 0.f : expf(red_m[w] - mx);
      l_run += red_l[w] * f;
#pragma unroll
      for (int i = 0; i < AG_MAX_D / RB_WAVE; ++i) {
        const int d = lane + i * RB_WAVE;
        if (d < head_dim) acc[i] += red_acc[w][d] * f;
      }
    }
  }
  if (sinks) l_run += expf(sinks[h] - m_run);          // a term of the denominator with no key and no value
  const float inv = sig_bias ? 1.0f : (l_run > 0.f ? 1.0f / l_run : 0.f);
  T* orow = out + ((size_t)t * n_heads + h) * head_dim;
#pragma unroll
  for (int i = 0; i < AG_MAX_D / RB_WAVE; ++i) {
    const int d = lane + i * RB_WAVE;
    if (d < head_dim) Num<T>::store(orow + d, acc[i] * inv);
  }
}

// The same for head sizes that are multiples of 4 (every size a real model has), with 16-byte loads
// (8-byte ones of bfloat16).  Scores: lane j takes key j of the page and walks its row four values at a
// time.  Weighted sum: the lanes are dealt in groups of G = the next power of two >= D / 4; group g takes
// the keys j = g, g + 64 / G, ... and lane c of a group the values 4 c .. 4 c + 3 of each, so that a
// group's load is one row of V in a piece; the groups' sums meet by shuffles once, after the last page.
// The scalar kernel above took 125 us for a decode step of 8 sequences at 530 keys of the 8B shape
// in float32 (every load instruction of its score loop touched 64 cache lines for 4 bytes each).
template <typename T>
struct Vec4;
template <>
struct Vec4<float> {
  static __device__ __forceinline__ float4 load(const float* p) { return *reinterpret_cast<const float4*>(p); }
};
template <>
struct Vec4<bf16_t> {
  static __device__ __forceinline__ float4 load(const bf16_t* p) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    return make_float4(bf16_bits_to_f32(v.x & 0xffffu), bf16_bits_to_f32(v.x >> 16), bf16_bits_to_f32(v.y & 0xffffu),
                       bf16_bits_to_f32(v.y >> 16));
  }
};

template <typename T>
__global__ __launch_bounds__(RB_WAVE * AG_MAX_WAVES) void attention_generic_vec_kernel(
    const T* __restrict__ q, const T* __restrict__ k_pages, const T* __restrict__ v_pages, T* __restrict__ out,
    const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ tok_seq,
    const int32_t* __restrict__ block_table, int bt_stride, int n_heads, int n_kv, int head_dim, float scale,
    int window, int group_lanes, const float* __restrict__ sinks, int keep_first, float softcap, int chunk,
    const float* __restrict__ sig_bias) {
  __shared__ __attribute__((aligned(16))) float qs[AG_MAX_D];
  __shared__ float ps_all[AG_MAX_WAVES][RB_PAGE];
  __shared__ float red_m[AG_MAX_WAVES], red_l[AG_MAX_WAVES];
  __shared__ __attribute__((aligned(16))) float red_acc[AG_MAX_WAVES][AG_MAX_D];
  const int t = blockIdx.x;
  const int h = blockIdx.y;
  const int lane = threadIdx.x & (RB_WAVE - 1);
  const int wave = threadIdx.x / RB_WAVE, n_waves = blockDim.x / RB_WAVE;
  float* ps = ps_all[wave];
  const int pos = tok_pos[t];
  const int kvh = h / (n_heads / n_kv);
  const int lo = first_visible(pos, window, chunk);
  const int32_t* pages = block_table + (size_t)tok_seq[t] * bt_stride;
  const int chunks = head_dim / 4;
  const int c = lane % group_lanes, g = lane / group_lanes, n_groups = RB_WAVE / group_lanes;
  const bool c_on = c < chunks;

  const T* qrow = q + ((size_t)t * n_heads + h) * head_dim;
  for (int d = threadIdx.x; d < head_dim; d += blockDim.x) qs[d] = Num<T>::load(qrow + d);
  __syncthreads();

  // sigmoid weights (sig_bias): a key's weight is sigmoid(score + sig_bias[h]) by itself, so the maximum stays 0, nothing is
  // rescaled and nothing divided
  const float sb = sig_bias ? sig_bias[h] : 0.f;
  float m_run = sig_bias ? 0.f : -INFINITY, l_run = 0.f;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  // the pages that hold visible keys: those of the kept first tokens that lie before the window's first page, then the
  // window's (every one of them holds at least one visible key)
  const int lo_page = lo / RB_PAGE;
  const int kept_pages = keep_first > 0 ? (keep_first + RB_PAGE - 1) / RB_PAGE : 0;
  const int n_first = kept_pages < lo_page ? kept_pages : lo_page;
  const int n_walk = n_first + pos / RB_PAGE - lo_page + 1;
  for (int walk = wave; walk < n_walk; walk += n_waves) {
    const int pg = walk < n_first ? walk : lo_page + walk - n_first;
    const size_t base = ((size_t)pages[pg] * n_kv + kvh) * RB_PAGE * head_dim;
    const int p = pg * RB_PAGE + lane;
    float s = -INFINITY;
    if (p <= pos && (p >= lo || p < keep_first)) {
      const T* krow = k_pages + base + (size_t)lane * head_dim;
      float d0 = 0.f, d1 = 0.f, d2 = 0.f, d3 = 0.f;
      for (int cc = 0; cc < chunks; ++cc) {
        const float4 kv = Vec4<T>::load(krow + 4 * cc);
        const float4 qv = *reinterpret_cast<const float4*>(qs + 4 * cc);
        d0 = fmaf(qv.x, kv.x, d0);
        d1 = fmaf(qv.y, kv.y, d1);
        d2 = fmaf(qv.z, kv.z, d2);
        d3 = fmaf(qv.w, kv.w, d3);
      }
      s = ((d0 + d1) + (d2 + d3)) * scale;
      if (softcap > 0.f) s = softcap * tanhf(s / softcap);
    }
    const float m_new = sig_bias ? 0.f : fmaxf(m_run, wave_max(s));      // finite: the page holds at least one valid key
    const float pexp = (s == -INFINITY) ? 0.f : (sig_bias ? 1.0f / (1.0f + expf(-(s + sb))) : expf(s - m_new));
    const float corr = (m_run == -INFINITY) ? 0.f : expf(m_run - m_new);
    l_run = l_run * corr + wave_sum(pexp);
    m_run = m_new;
    ps[lane] = pexp;                                    // this wave's alone; a wave's LDS accesses complete in order
    __builtin_amdgcn_wave_barrier();
    const int j_lo = (pg * RB_PAGE < lo && pg * RB_PAGE >= keep_first) ? lo - pg * RB_PAGE : 0;      // keys between carry weight 0
    const int j_hi = (pg * RB_PAGE + RB_PAGE - 1 > pos) ? pos - pg * RB_PAGE : RB_PAGE - 1;
    acc.x *= corr;
    acc.y *= corr;
    acc.z *= corr;
    acc.w *= corr;
    if (c_on) {
      const T* vcol = v_pages + base + 4 * c;
      for (int j = j_lo + g; j <= j_hi; j += n_groups) {
        const float4 vv = Vec4<T>::load(vcol + (size_t)j * head_dim);
        const float w = ps[j];
        acc.x = fmaf(w, vv.x, acc.x);
        acc.y = fmaf(w, vv.y, acc.y);
        acc.z = fmaf(w, vv.z, acc.z);
        acc.w = fmaf(w, vv.w, acc.w);
      }
    }
  }
  // the groups' sums meet in group 0
  for (int o = group_lanes; o < RB_WAVE; o <<= 1) {
    acc.x += __shfl_xor(acc.x, o, RB_WAVE);
    acc.y += __shfl_xor(acc.y, o, RB_WAVE);
    acc.z += __shfl_xor(acc.z, o, RB_WAVE);
    acc.w += __shfl_xor(acc.w, o, RB_WAVE);
  }
  const bool owner = g == 0 && c_on;
  // ---- the waves' states into one (a wave without pages holds m = -inf, l = 0, acc = 0)
  if (n_waves > 1) {
    if (lane == 0) {
      red_m[wave] = m_run;
      red_l[wave] = l_run;
    }
    if (owner) *reinterpret_cast<float4*>(&red_acc[wave][4 * c]) = acc;
    __syncthreads();
    if (wave != 0) return;
    float mx = red_m[0];
    for (int w = 1; w < n_waves; ++w) mx = fmaxf(mx, red_m[w]);
    m_run = mx;
    l_run = 0.f;
    acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int w = 0; w < n_waves; ++w) {
      const float f = (red_m[w] == -INFINITY) ? 0.f : expf(red_m[w] - mx);
      l_run += red_l[w] * f;
      if (owner) {
        const float4 a = *reinterpret_cast<const float4*>(&red_acc[w][4 * c]);
        acc.x += a.x * f;
        acc.y += a.y * f;
        acc.z += a.z * f;
        acc.w += a.w * f;
      }
    }
  }
  if (owner) {
    if (sinks) l_run += expf(sinks[h] - m_run);        // a term of the denominator with no key and no value
    const float inv = sig_bias ? 1.0f : (l_run > 0.f ? 1.0f / l_run : 0.f);
    T* orow = out + ((size_t)t * n_heads + h) * head_dim + 4 * c;
    Num<T>::store(orow + 0, acc.x * inv);
    Num<T>::store(orow + 1, acc.y * inv);
    Num<T>::store(orow + 2, acc.z * inv);
    Num<T>::store(orow + 3, acc.w * inv);
  }
}

// x, for comparisons that are made where they stand: made ahead of a loop, they hold more scalar registers than there are.
__device__ __forceinline__ int here(int x) {
  asm volatile("" : "+s"(x));
  return x;
}

// Float32 attention on the float32 MFMA (16x16x4: float32 inputs, products and sums), for head sizes that are multiples of 4 up to
// 128.  The 16 columns of the MFMAs are queries: the heads that share a key/value head, of one token or of as many consecutive
// tokens as fit, so that a key is read once for all of them.  Scores are K Q^T (a lane takes one key's row, 16 bytes at a time, and
// four MFMAs use the four floats of it), so that a lane ends up with 4 keys' weights of one query, which is what the second
// product, V^T P^T, takes as its operand as they are; V's rows are dealt to the lanes NB numbers at a time (MFMA dt works on the
// numbers NB r + dt of a head for its row r), so that they come with wide loads and leave as pieces of rows.  The waves of a workgroup
// share the keys, 32 at a time, and merge through LDS at the end.  Softmax, its running maximum, caps, sinks, windows, kept first
// keys, chunks and sigmoid weights as in the kernels above.
// A score is four sums (of every fourth number), a unit of 32 keys has sums of its own, 16 / NB of them side by side, which are added up
// as a tree before they meet the running ones, and so are its weights: one sum for everything had twice the error. Relative error of
// the outputs, 24 heads of 128 at 131 to 512 keys / one token at 8,000: 3.2e-7 / 6.8e-7 with one sum, 1.5e-7 / 2.4e-7 now, 1.7e-7 / 4.4e-7 in
// the kernel above; heads of 24: 1.7e-7 / 6.9e-7, 1.2e-7 / 2.3e-7 and 1.3e-7 / 2.8e-7.
// Bound by the MFMAs for prompts (2 x 32 cycles for 16 keys, 16 queries and 4 numbers) and by a chain of loads in single-token steps.
// Measured beside the kernel above (a lane per key on the vector units; caches as a step finds them: what the step wrote is not in a
// workgroup's own, keys of earlier steps are in none), 24 heads of 128 on 8: four prompts of 131 to 512 tokens 608 -> 130 us a layer, one
// of 8 / 30 / 100 tokens 7.0 / 10.1 / 28 -> 8.0 / 8.2 / 12.7; single tokens at 150 / 1,000 keys: one sequence 22 / 51 -> 13.5 / 42, 16 27 / 88 -> 16 / 70,
// 64 55 / 246 -> 39 / 162.  32 heads on 32, 64 sequences 159 / 784 -> 133 / 418.
// ONE: a block is one token's, and where tokens and kv heads leave the GPU empty up to MAX_SHARING workgroups share its keys: as many as
// have a unit of 32 keys for each of their 8 waves, known from the token's position, so that short contexts stay with one and pay nothing.
// Whoever of them is done last adds up (no second launch, no waiting).  24 heads of 128 on 8, one workgroup / shared by up to 4: one token at
// 250 / 280 / 400 / 1,000 / 4,000 keys 15.0 / 17.3 / 21.5 / 42.9 / 139.7 -> 14.6 / 14.9 / 16.3 / 18.6 / 46.3 us (28.3 by 8), four at 1,000 44.5 -> 19.9.
constexpr int MAX_SHARING = 8;      // workgroups of a token's keys
template <int NB, bool ONE>
__global__ __launch_bounds__(RB_WAVE * AG_MAX_WAVES) void attention_f32_mfma_kernel(
    const float* __restrict__ q, const float* __restrict__ k_pages, const float* __restrict__ v_pages, float* __restrict__ out,
    const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ tok_seq, const int32_t* __restrict__ block_table, int bt_stride,
    int n_tokens, int n_heads, int n_kv, int head_dim, float scale, int window, const float* __restrict__ sinks, int keep_first,
    float softcap, int chunk, const float* __restrict__ sig_bias, int tokens_per_block, int head_chunks, int32_t* __restrict__ arrived,
    float* __restrict__ parts) {
  constexpr int VW = NB < 4 ? NB : 4;                  // floats of a load of V
  constexpr int CHAINS = 16 / NB;                      // the shorter a head, the more sums a unit's values go into
  constexpr int LD = 16 * NB + 4;                      // a query's row in LDS: outputs, then maximum and sum
  extern __shared__ __attribute__((aligned(16))) float merged[];      // [waves][16][LD]
  const int lane = threadIdx.x & (RB_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / RB_WAVE), n_waves = blockDim.x / RB_WAVE;
  const int col = lane & 15, g = lane >> 4;
  const int group = n_heads / n_kv;
  const int kvh = blockIdx.y / head_chunks, first = (blockIdx.y % head_chunks) * 16;
  const int h_count = group - first < 16 ? group - first : 16;
  const int h0 = kvh * group + first;
  // late tokens first: they have the most keys
  const int t0 = (gridDim.x - 1 - blockIdx.x) * (ONE ? 1 : tokens_per_block);
  const int t1 = ONE ? t0 + 1 : t0 + tokens_per_block < n_tokens ? t0 + tokens_per_block : n_tokens;
  const int t = ONE ? t0 : t0 + col / h_count, h = ONE ? h0 + col : h0 + col % h_count;
  const bool on = ONE ? col < h_count : t < t1;
  // The block's tokens, a lane each (one trip to memory), and where a run of consecutive positions of one sequence starts among them.
  const int count = t1 - t0;
  const int l_seq = lane < count ? tok_seq[t0 + lane] : -1, l_pos = lane < count ? tok_pos[t0 + lane] : -1;
  const int seq_before = __shfl_up(l_seq, 1, RB_WAVE), pos_before = __shfl_up(l_pos, 1, RB_WAVE);
  unsigned long long starts = __ballot(lane == 0 || lane == count || (lane < count && (l_seq != seq_before || l_pos != pos_before + 1)));
  const int my_pos = ONE ? __builtin_amdgcn_readfirstlane(l_pos) : __shfl(l_pos, t - t0, RB_WAVE);      // (of a column in use)
  const int my_lo = on ? first_visible(my_pos, window, chunk) : 0;

  f32x4_t qv[NB];
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    qv[c] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    if (on && 16 * c + 4 * g < head_dim)
      qv[c] = *reinterpret_cast<const f32x4_t*>(q + ((size_t)t * n_heads + h) * head_dim + 16 * c + 4 * g);
  }
  const float sb = sig_bias && on ? sig_bias[h] : 0.f;

  // Run after run: almost always the whole block is one.  Each starts anew and leaves with its own columns only, so that nothing of
  // another sequence comes into a query's sums, and tokens may come in any order.
  bool in_use = false;                        // what the waves share in LDS
  for (int seg = t0, end; seg < t1; seg = end) {
    starts &= starts - 1;
    end = ONE ? t1 : t0 + __builtin_ctzll(starts);
    const int seq = __builtin_amdgcn_readlane(l_seq, seg - t0);
    const int32_t* pages = block_table + (size_t)seq * bt_stride;
    const int hi = __builtin_amdgcn_readlane(l_pos, end - 1 - t0);
    const int lo = first_visible(__builtin_amdgcn_readlane(l_pos, seg - t0), window, chunk);
    const bool mine = ONE ? on : t >= seg && t < end;
    auto sees = [&](int key) { return mine && key <= my_pos && (key >= my_lo || key < keep_first); };
    // A weight of 0 does not take an infinity or a NaN out of a matrix product.  One token's queries see the same keys: the values of
    // others become zeros.
    auto hidden = [&](int key) { return key > hi || (key < lo && key >= keep_first); };
    f32x4_t acc[NB];
#pragma unroll
    for (int d = 0; d < NB; ++d) acc[d] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    float m_run = sig_bias ? 0.f : -INFINITY, l_run = 0.f;
    const int lo_unit = lo / 32;
    const int kept = keep_first > 0 ? (keep_first + 31) / 32 : 0;
    const int n_first = kept < lo_unit ? kept : lo_unit;
    const int n_walk = hi < 0 ? 0 : n_first + hi / 32 - lo_unit + 1;      // (without a position there are no keys)
    // One token's keys: as many workgroups as its waves have keys for share them, the others are done (all of a token know the same).
    const int needed = (n_walk + n_waves - 1) / n_waves;
    const int sharing = !ONE || needed <= 1 ? 1 : needed < (int)gridDim.z ? needed : (int)gridDim.z;
    const int part = ONE ? blockIdx.z : 0;
    if (part >= sharing) return;
    for (int walk = wave * sharing + part; walk < n_walk; walk += n_waves * sharing) {
      const int key0 = 32 * (walk < n_first ? walk : lo_unit + walk - n_first);
      const size_t base = ((size_t)pages[key0 / RB_PAGE] * n_kv + kvh) * RB_PAGE * head_dim + (size_t)(key0 % RB_PAGE) * head_dim;
      // keys behind the last one are not written yet: the last one's numbers stand in for them, with weight 0
      f32x4_t kf[2][NB];
      float vf[2][4][NB];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int kr = (key0 + 16 * b + col < hi ? key0 + 16 * b + col : hi) - key0;
        const float* krow = k_pages + base + (size_t)kr * head_dim + 4 * g;
#pragma unroll
        for (int c = 0; c < NB; ++c) {
          kf[b][c] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
          if (16 * c + 4 * g < head_dim) kf[b][c] = *reinterpret_cast<const f32x4_t*>(krow + 16 * c);
        }
      }
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = key0 + 16 * b + 4 * g + i;
          const float* vrow = v_pages + base + (size_t)((key < hi ? key : hi) - key0) * head_dim + NB * col;
#pragma unroll
          for (int d = 0; d < NB; d += VW) {
            if (NB * col + d < head_dim) {
              if (VW == 4) *reinterpret_cast<f32x4_t*>(&vf[b][i][d]) = *reinterpret_cast<const f32x4_t*>(vrow + d);
              else *reinterpret_cast<float2*>(&vf[b][i][d]) = *reinterpret_cast<const float2*>(vrow + d);
            } else {
#pragma unroll
              for (int e = 0; e < VW; ++e) vf[b][i][d + e] = 0.f;
            }
          }
        }
      if (ONE && (key0 + 31 > hi || key0 < lo)) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (hidden(key0 + 16 * b + 4 * g + i)) {
#pragma unroll
              for (int d = 0; d < NB; ++d) vf[b][i][d] = 0.f;
            }
      }
      f32x4_t sc[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        f32x4_t part[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) part[i] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < NB; ++c)
#pragma unroll
          for (int i = 0; i < 4; ++i) part[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[b][c][i], qv[c][i], part[i], 0, 0, 0);
        sc[b] = (part[0] + part[1]) + (part[2] + part[3]);
      }
      float top = -INFINITY;
      bool in_part = false;                   // some query of the run does not see one of these keys
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = key0 + 16 * b + 4 * g + i;
          float s = sc[b][i] * scale;
          if (softcap > 0.f) s = softcap * tanhf(s / softcap);
          const bool seen = sees(key);
          s = seen ? s : -INFINITY;
          if (!ONE) in_part |= mine && !seen;
          sc[b][i] = s;
          top = fmaxf(top, s);
        }
      top = fmaxf(top, __shfl_xor(top, 16, RB_WAVE));
      top = fmaxf(top, __shfl_xor(top, 32, RB_WAVE));
      const float m_new = sig_bias ? 0.f : fmaxf(m_run, top);
      const float corr = m_run == -INFINITY ? 0.f : expf(m_run - m_new);      // nothing seen yet: nothing to rescale
      m_run = m_new;
      l_run *= corr;
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float s = sc[b][i];
          sc[b][i] = s == -INFINITY ? 0.f : (sig_bias ? 1.0f / (1.0f + expf(-(s + sb))) : expf(s - m_new));
        }
      l_run += ((sc[0][0] + sc[0][1]) + (sc[0][2] + sc[0][3])) + ((sc[1][0] + sc[1][1]) + (sc[1][2] + sc[1][3]));
#pragma unroll
      for (int d = 0; d < NB; ++d) acc[d] *= corr;
      // Several tokens': where a query does not see all of these keys and a value is an infinity or a NaN, every query adds up the
      // keys that it sees, by itself.
      bool bad = false;
      if (!ONE && __any(in_part)) {
        float zero = 0.f;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int d = 0; d < NB; ++d) zero = fmaf(vf[b][i][d], 0.f, zero);
        bad = __any(zero != 0.f);
      }
      if (bad) {
#pragma unroll 1
        for (int kk = 0; kk < 32; ++kk) {
          const f32x4_t four = kk < 16 ? sc[0] : sc[1];
          const int i = kk & 3;
          const float p = __shfl(i == 0 ? four[0] : i == 1 ? four[1] : i == 2 ? four[2] : four[3], (kk & 12) * 4 + col, RB_WAVE);
          if (!sees(key0 + kk)) continue;
          const float* vrow = v_pages + base + (size_t)kk * head_dim + 4 * NB * g;
          const int left = here(head_dim) - 4 * NB * g;
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int d = 0; d < NB; d += VW)
              if (NB * j + d < left) {
                float v[VW];
                if (VW == 4) *reinterpret_cast<f32x4_t*>(v) = *reinterpret_cast<const f32x4_t*>(vrow + NB * j + d);
                else *reinterpret_cast<float2*>(v) = *reinterpret_cast<const float2*>(vrow + NB * j + d);
#pragma unroll
                for (int e = 0; e < VW; ++e) acc[d + e][j] = fmaf(p, v[e], acc[d + e][j]);
              }
        }
      } else {
        f32x4_t unit[CHAINS][NB];
#pragma unroll
        for (int n = 0; n < CHAINS; ++n)
#pragma unroll
          for (int d = 0; d < NB; ++d) unit[n][d] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int d = 0; d < NB; ++d) {
              f32x4_t& sum = unit[(4 * b + i) % CHAINS][d];
              sum = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[b][i][d], sc[b][i], sum, 0, 0, 0);
            }
#pragma unroll
        for (int n = CHAINS / 2; n > 0; n /= 2)
#pragma unroll
          for (int m = 0; m < n; ++m)
#pragma unroll
            for (int d = 0; d < NB; ++d) unit[m][d] += unit[m + n][d];
#pragma unroll
        for (int d = 0; d < NB; ++d) acc[d] += unit[0][d];
      }
    }
    l_run += __shfl_xor(l_run, 16, RB_WAVE);
    l_run += __shfl_xor(l_run, 32, RB_WAVE);

    // lane holds, for query col, the numbers NB (4 g + j) + d of the head
    const int mine_of = (n_walk - part + sharing - 1) / sharing;           // units of this workgroup
    const int at_work = mine_of > n_waves ? n_waves : mine_of;    // waves that had keys: the first ones
    if (at_work <= 1 && sharing == 1) {
      if (!mine || wave > 0) continue;
      if (sinks) l_run += expf(sinks[h] - m_run);
      const float inv = sig_bias ? 1.0f : (l_run > 0.f ? 1.0f / l_run : 0.f);
      float* orow = out + ((size_t)t * n_heads + h) * head_dim + 4 * NB * g;
      const int left = here(head_dim) - 4 * NB * g;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int d = 0; d < NB; ++d)
          if (NB * j + d < left) orow[NB * j + d] = acc[d][j] * inv;
      continue;
    }
    if (in_use) __syncthreads();              // the run before has been read
    in_use = true;
    float* row = merged + ((size_t)wave * 16 + col) * LD;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int d = 0; d < NB; ++d) row[NB * (4 * g + j) + d] = acc[d][j];
    if (g == 0) {
      row[16 * NB] = m_run;
      row[16 * NB + 1] = l_run;
    }
    __syncthreads();
    // every thread finishes a few numbers of a query: the waves' sums under their common maximum, in the order of the waves
    const int first_col = (seg - t0) * h_count, queries = (end - seg) * h_count;
    for (int idx = threadIdx.x; idx < queries * head_dim; idx += blockDim.x) {
      const int q_of = idx / head_dim, d = idx - q_of * head_dim, cc = first_col + q_of;
      const int hh = h0 + cc % h_count;
      const float* src = merged + (size_t)cc * LD;
      float mx = -INFINITY;
      for (int w = 0; w < at_work; ++w) mx = fmaxf(mx, src[(size_t)w * 16 * LD + 16 * NB]);
      float l = 0.f, o = 0.f;
      for (int w = 0; w < at_work; ++w) {
        const float mw = src[(size_t)w * 16 * LD + 16 * NB];
        const float f = mw == -INFINITY ? 0.f : expf(mw - mx);
        l += src[(size_t)w * 16 * LD + 16 * NB + 1] * f;
        o += src[(size_t)w * 16 * LD + d] * f;
      }
      if (sharing > 1) {
        float* dst = parts + (((size_t)t0 * n_heads + hh) * gridDim.z + part) * (head_dim + 2);
        __hip_atomic_store(dst + d, o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (d == 0) {
          __hip_atomic_store(dst + head_dim, mx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(dst + head_dim + 1, l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        continue;
      }
      if (sinks) l += expf(sinks[hh] - mx);
      const float inv = sig_bias ? 1.0f : (l > 0.f ? 1.0f / l : 0.f);
      out[((size_t)(t0 + cc / h_count) * n_heads + hh) * head_dim + d] = o * inv;
    }
    if (ONE && sharing > 1) {
      // Whoever is done last adds up what all have left, in their order; nobody waits for another.  What they leave goes through to
      // where every workgroup sees it (atomic stores and loads of the device's scope) and has arrived before its wave counts: a fence
      // would write back the whole L2 instead, 10 to 20 us with 128 workgroups.
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      int32_t* count = arrived + (size_t)t0 * gridDim.y + blockIdx.y;
      if (threadIdx.x == 0) {
        const bool last = __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == sharing - 1;
        if (last) __hip_atomic_store(count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);      // for the next launch
        merged[0] = last ? 1.f : 0.f;
      }
      __syncthreads();
      if (merged[0] == 0.f) return;
      asm volatile("" ::: "memory");
      for (int idx = threadIdx.x; idx < h_count * head_dim; idx += blockDim.x) {
        const int hh = h0 + idx / head_dim, d = idx % head_dim;
        const float* src = parts + ((size_t)t0 * n_heads + hh) * gridDim.z * (head_dim + 2);
        float top[MAX_SHARING], sum[MAX_SHARING], value[MAX_SHARING];
#pragma unroll
        for (int w = 0; w < MAX_SHARING; ++w) {
          const float* from = src + (size_t)(w < sharing ? w : sharing - 1) * (head_dim + 2);
          top[w] = __hip_atomic_load(from + head_dim, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          sum[w] = __hip_atomic_load(from + head_dim + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          value[w] = __hip_atomic_load(from + d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < MAX_SHARING; ++w) mx = fmaxf(mx, top[w]);
        float l = 0.f, o = 0.f;
#pragma unroll
        for (int w = 0; w < MAX_SHARING; ++w)
          if (w < sharing) {
            const float f = top[w] == -INFINITY ? 0.f : expf(top[w] - mx);
            l += sum[w] * f;
            o += value[w] * f;
          }
        if (sinks) l += expf(sinks[hh] - mx);
        const float inv = sig_bias ? 1.0f : (l > 0.f ? 1.0f / l : 0.f);
        out[((size_t)t0 * n_heads + hh) * head_dim + d] = o * inv;
      }
    }
  }
}

struct AttentionF32 {
  const float *q, *k_pages, *v_pages;
  float* out;
  const int32_t *tok_pos, *tok_seq, *block_table;
  int bt_stride, n_tokens, n_heads, n_kv, head_dim;
  float scale;
  int window;
  const float* sinks;
  int keep_first;
  float softcap;
  int chunk;
  const float* sig_bias;
  int n_seqs;            // 0: not known
  int n_splits;          // workgroups that may share a token's keys
  void* workspace;
};

template <int NB, bool ONE>
static int launch_attention_f32_blocks(const AttentionF32& a, int per_block, int chunks, hipStream_t s) {
  const long long cus = rb_compute_units();
  const long long blocks = ((long long)a.n_tokens + per_block - 1) / per_block;
  int n_waves = 1;
  while (n_waves < AG_MAX_WAVES && blocks * a.n_kv * chunks * n_waves < 8 * cus) n_waves *= 2;
  RB_REQUIRE((long long)a.n_kv * chunks <= 65535, "rb_attention_generic: too many heads %d", a.n_heads);
  const size_t lds = n_waves > 1 ? (size_t)n_waves * 16 * (16 * NB + 4) * sizeof(float) : 0;
  auto kern = attention_f32_mfma_kernel<NB, ONE>;
  static bool configured = false;
  if (!configured) {
    const size_t most = (size_t)AG_MAX_WAVES * 16 * (16 * NB + 4) * sizeof(float);
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)most);
    RB_REQUIRE(e == hipSuccess, "rb_attention_generic: cannot reserve %zu bytes of LDS: %s", most, hipGetErrorString(e));
    configured = true;
  }
  const int splits = ONE && n_waves > 1 ? a.n_splits : 1;
  int32_t* arrived = (int32_t*)a.workspace;
  float* parts = a.workspace ? (float*)a.workspace + (size_t)a.n_tokens * a.n_heads : nullptr;
  kern<<<dim3((unsigned)blocks, (unsigned)(a.n_kv * chunks), (unsigned)splits), RB_WAVE * n_waves, lds, s>>>(
      a.q, a.k_pages, a.v_pages, a.out, a.tok_pos, a.tok_seq, a.block_table, a.bt_stride, a.n_tokens, a.n_heads, a.n_kv, a.head_dim,
      a.scale, a.window, a.sinks, a.keep_first, a.softcap, a.chunk, a.sig_bias, per_block, chunks, arrived, parts);
  return 0;
}

template <int NB>
static int launch_attention_f32(const AttentionF32& a, hipStream_t s) {
  const int group = a.n_heads / a.n_kv, chunks = (group + 15) / 16;
  // How many tokens share a block's 16 columns: as many as fit where one token a block (whose other columns are idle) would make more
  // blocks than the GPU has room for.  A block over a boundary takes its sequences one after another, so with several of them that is
  // four blocks a compute unit, with one sequence one (24 heads of 128 on 8, one prompt of 100 tokens: 21.4 us with one token a block,
  // 12.7 with 5; four of 16: 8.7 and 13; four of 40: 14.0 and 10.6), and never in a single-token step (32 sequences at 150 / 1,000 keys, 32
  // heads of 128: 66 / 240 us with one token a block, 177 / 630 with 16).
  const long long blocks_of_one = (long long)a.n_tokens * a.n_kv * chunks;
  const bool share = a.n_seqs != a.n_tokens && blocks_of_one >= (a.n_seqs == 1 ? 1 : 4) * rb_compute_units();
  const int per_block = share && group < 16 ? 16 / group : 1;
  if (per_block == 1) return launch_attention_f32_blocks<NB, true>(a, 1, chunks, s);
  return launch_attention_f32_blocks<NB, false>(a, per_block, chunks, s);
}

static int g_attention_vec = 1;
extern "C" void rb_tune_attention_vec(int on) { g_attention_vec = on; }      // experiments and tests: 0 = the scalar kernel for every head size, 2 = not the float32 matrix cores

extern "C" int rb_attention_generic(const void* q, const void* k_pages, const void* v_pages, void* out, int dtype,
                                    const int32_t* tok_pos, const int32_t* tok_seq, const int32_t* block_table,
                                    int bt_stride, int n_tokens, int n_heads, int n_kv_heads, int head_dim,
                                    float scale, int window, void* stream) {
  return rb_attention_generic_sinks(q, k_pages, v_pages, out, dtype, tok_pos, tok_seq, block_table, bt_stride, n_tokens,
                                    n_heads, n_kv_heads, head_dim, scale, window, nullptr, stream);
}

// The same with a sink per query head (sinks float32 [Hq], null: none): the softmax's denominator also holds
// exp(sink), a score that is not scaled and belongs to no key and no value.  v_pages may be k_pages.
extern "C" int rb_attention_generic_sinks(const void* q, const void* k_pages, const void* v_pages, void* out, int dtype,
                                          const int32_t* tok_pos, const int32_t* tok_seq, const int32_t* block_table,
                                          int bt_stride, int n_tokens, int n_heads, int n_kv_heads, int head_dim,
                                          float scale, int window, const float* sinks, void* stream) {
  RB_RECORDED(rb_attention_generic_sinks(q, k_pages, v_pages, out, dtype, tok_pos, tok_seq, block_table, bt_stride, n_tokens,
                                         n_heads, n_kv_heads, head_dim, scale, window, sinks, stream));
  return rb_attention_generic_opts(q, k_pages, v_pages, out, dtype, tok_pos, tok_seq, block_table, bt_stride, n_tokens, n_heads,
                                   n_kv_heads, head_dim, scale, window, 0, 0.0f, sinks, stream);
}

// The same with two more choices.  keep_first (with a window): the first keep_first keys of a sequence stay visible behind
// the window, a query at position i seeing j <= i with i - j < window or j < keep_first.  softcap > 0: a score s becomes
// softcap * tanh(s / softcap) after the scale and before the softmax.
extern "C" int rb_attention_generic_opts(const void* q, const void* k_pages, const void* v_pages, void* out, int dtype,
                                         const int32_t* tok_pos, const int32_t* tok_seq, const int32_t* block_table,
                                         int bt_stride, int n_tokens, int n_heads, int n_kv_heads, int head_dim,
                                         float scale, int window, int keep_first, float softcap, const float* sinks,
                                         void* stream) {
  RB_RECORDED(rb_attention_generic_opts(q, k_pages, v_pages, out, dtype, tok_pos, tok_seq, block_table, bt_stride, n_tokens,
                                        n_heads, n_kv_heads, head_dim, scale, window, keep_first, softcap, sinks, stream));
  return rb_attention_generic_chunked(q, k_pages, v_pages, out, dtype, tok_pos, tok_seq, block_table, bt_stride, n_tokens, n_heads,
                                      n_kv_heads, head_dim, scale, window, keep_first, softcap, sinks, 0, nullptr, stream);
}

// The same with two more.  chunk > 0: a query at position i sees the keys j <= i with i / chunk == j / chunk only (beside
// what the window says).  sig_bias (float32 [Hq], null: softmax): a visible key's weight is sigmoid(score + sig_bias[h]), and
// the weights are not normalised over the keys (a sink then has no meaning and must be null).
extern "C" int rb_attention_generic_chunked(const void* q, const void* k_pages, const void* v_pages, void* out, int dtype,
                                            const int32_t* tok_pos, const int32_t* tok_seq, const int32_t* block_table,
                                            int bt_stride, int n_tokens, int n_heads, int n_kv_heads, int head_dim,
                                            float scale, int window, int keep_first, float softcap, const float* sinks, int chunk,
                                            const float* sig_bias, void* stream) {
  RB_RECORDED(rb_attention_generic_chunked(q, k_pages, v_pages, out, dtype, tok_pos, tok_seq, block_table, bt_stride, n_tokens,
                                           n_heads, n_kv_heads, head_dim, scale, window, keep_first, softcap, sinks, chunk, sig_bias,
                                           stream));
  return rb_attention_generic_steps(q, k_pages, v_pages, out, dtype, tok_pos, tok_seq, block_table, bt_stride, n_tokens, n_heads,
                                    n_kv_heads, head_dim, scale, window, keep_first, softcap, sinks, chunk, sig_bias, 0, 1, nullptr,
                                    stream);
}

// The same, told how many sequences the tokens are of (0: not known; it decides between kernels, not what is computed), and how many
// workgroups may share the keys of a token where every sequence has one (1: none).  workspace, where that is more than one:
// n_tokens * n_heads counters, zeros before and after, then n_tokens * n_heads * n_splits * (head_dim + 2) floats.
extern "C" int rb_attention_generic_steps(const void* q, const void* k_pages, const void* v_pages, void* out, int dtype,
                                          const int32_t* tok_pos, const int32_t* tok_seq, const int32_t* block_table,
                                          int bt_stride, int n_tokens, int n_heads, int n_kv_heads, int head_dim,
                                          float scale, int window, int keep_first, float softcap, const float* sinks, int chunk,
                                          const float* sig_bias, int n_seqs, int n_splits, void* workspace, void* stream) {
  RB_RECORDED(rb_attention_generic_steps(q, k_pages, v_pages, out, dtype, tok_pos, tok_seq, block_table, bt_stride, n_tokens,
                                         n_heads, n_kv_heads, head_dim, scale, window, keep_first, softcap, sinks, chunk, sig_bias,
                                         n_seqs, n_splits, workspace, stream));
  RB_REQUIRE(keep_first >= 0 && softcap >= 0.f && chunk >= 0, "rb_attention_generic: negative keep_first, softcap or chunk");
  RB_REQUIRE(sig_bias == nullptr || sinks == nullptr, "rb_attention_generic: a sink belongs to the softmax");
  RB_REQUIRE(n_tokens >= 0 && n_heads > 0 && n_kv_heads > 0 && n_heads % n_kv_heads == 0,
             "rb_attention_generic: bad head counts Hq=%d Hk=%d", n_heads, n_kv_heads);
  RB_REQUIRE(head_dim > 0 && head_dim <= AG_MAX_D, "rb_attention_generic: head_dim %d not supported (at most %d)", head_dim,
             AG_MAX_D);
  RB_REQUIRE(n_heads <= 65535, "rb_attention_generic: too many heads %d", n_heads);
  RB_REQUIRE(window >= 0, "rb_attention_generic: negative window");
  RB_REQUIRE(n_splits >= 1 && n_splits <= MAX_SHARING && (n_splits == 1 || workspace != nullptr),
             "rb_attention_generic: %d workgroups for a token's keys need a workspace and are at most %d", n_splits, MAX_SHARING);
  RB_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 3) == 0, "rb_attention_generic: the workspace is not aligned");
  if (n_tokens == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const bool wide = ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k_pages) | reinterpret_cast<uintptr_t>(v_pages)) & 15) == 0;
  if (dtype == RB_F32 && head_dim % 4 == 0 && head_dim <= 128 && wide && g_attention_vec == 1) {
    const AttentionF32 a = {(const float*)q, (const float*)k_pages, (const float*)v_pages, (float*)out, tok_pos, tok_seq, block_table,
                            bt_stride, n_tokens, n_heads, n_kv_heads, head_dim, scale, window, sinks, keep_first, softcap, chunk, sig_bias, n_seqs, n_splits, workspace};
    const int rc = head_dim <= 32 ? launch_attention_f32<2>(a, s) : head_dim <= 64 ? launch_attention_f32<4>(a, s) : launch_attention_f32<8>(a, s);
    if (rc) return rc;
    RB_LAUNCH_CHECK();
    return 0;
  }
  dim3 grid(n_tokens, n_heads);
  // waves per (token, head): enough to give every SIMD of the GPU two waves, at most 8
  int n_waves = 1;
  while (n_waves < AG_MAX_WAVES && (long long)n_tokens * n_heads * n_waves < 8LL * rb_compute_units()) n_waves *= 2;
  const int threads = RB_WAVE * n_waves;
  if (head_dim % 4 == 0 && head_dim <= AG_MAX_D_VEC && g_attention_vec) {
    int group_lanes = 1;
    while (group_lanes < head_dim / 4) group_lanes *= 2;
    RB_REQUIRE(dtype == RB_F32 || dtype == RB_BF16, "rb_attention_generic: unknown dtype %d", dtype);
    if (dtype == RB_F32)
      attention_generic_vec_kernel<float><<<grid, threads, 0, s>>>((const float*)q, (const float*)k_pages,
                                                                  (const float*)v_pages, (float*)out, tok_pos, tok_seq,
                                                                  block_table, bt_stride, n_heads, n_kv_heads, head_dim,
                                                                  scale, window, group_lanes, sinks, keep_first, softcap,
                                                                  chunk, sig_bias);
    else
      attention_generic_vec_kernel<bf16_t><<<grid, threads, 0, s>>>((const bf16_t*)q, (const bf16_t*)k_pages,
                                                                   (const bf16_t*)v_pages, (bf16_t*)out, tok_pos,
                                                                   tok_seq, block_table, bt_stride, n_heads, n_kv_heads,
                                                                   head_dim, scale, window, group_lanes, sinks, keep_first, softcap, chunk,
                                                                   sig_bias);
    RB_LAUNCH_CHECK();
    return 0;
  }
  if (dtype == RB_F32)
    attention_generic_kernel<float><<<grid, threads, 0, s>>>((const float*)q, (const float*)k_pages,
                                                            (const float*)v_pages, (float*)out, tok_pos, tok_seq,
                                                            block_table, bt_stride, n_heads, n_kv_heads, head_dim,
                                                            scale, window, sinks, keep_first, softcap, chunk, sig_bias);
  else if (dtype == RB_BF16)
    attention_generic_kernel<bf16_t><<<grid, threads, 0, s>>>((const bf16_t*)q, (const bf16_t*)k_pages,
                                                             (const bf16_t*)v_pages, (bf16_t*)out, tok_pos,
                                                             tok_seq, block_table, bt_stride, n_heads, n_kv_heads,
                                                             head_dim, scale, window, sinks, keep_first, softcap, chunk, sig_bias);
  else
    RB_REQUIRE(false, "rb_attention_generic: unknown dtype %d", dtype);
  RB_LAUNCH_CHECK();
  return 0;
}
