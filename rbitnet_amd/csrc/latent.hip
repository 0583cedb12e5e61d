// Attention through a latent: every token leaves one vector c of kv_rank numbers in the cache, and each head's
// keys and values are products of c with matrices of that head.  The products are moved to the query's side, so that
// attention runs over the cached latents themselves, as one key/value head of size kv_rank that all query heads share:
//   score = q . (Wk c) = (Wk^T q) . c,      out = Wv (sum_j p_j c_j)
// Here: the RMS norms of the two down-projections with the cache write, and the per-head products on either side
// of attention.  float32 arithmetic; storage float32 or bfloat16.
#include <math.h>

#include "api.h"
#include "common.h"
#include "decode_combine.h"
#include "mfma.h"

// proj [T, stride] float32 holds, per token, q_rank numbers at column 0 and kv_rank numbers at column kv_col.
// cq[t] = rmsnorm(proj[t, 0:q_rank]) * q_gain; c = rmsnorm(proj[t, kv_col:kv_col + kv_rank]) * kv_gain goes into the
// token's place of the cache pages [pages, 1, 64, kv_rank].  Either half may be absent (rank 0).
template <typename TC>
__global__ void latent_norm_store_kernel(const float* __restrict__ proj, size_t stride, int q_rank,
                                         const float* __restrict__ q_gain, TC* __restrict__ cq, int kv_col, int kv_rank,
                                         const float* __restrict__ kv_gain, TC* __restrict__ pages, int page_width,
                                         const int32_t* __restrict__ tok_pos, const int32_t* __restrict__ tok_seq,
                                         const int32_t* __restrict__ block_table, int bt_stride, float eps, int rot_col = 0,
                                         int rot = 0, const float* __restrict__ cos_t = nullptr,
                                         const float* __restrict__ sin_t = nullptr, int style = 0) {
  __shared__ float scratch[16];
  // the two norms are two workgroups of a token: one behind the other they were a chain of four trips to memory (four tokens,
  // ranks of 768 and 96: 6.0 -> 4.2 us)
  const int t = blockIdx.x;
  const float* row = proj + (size_t)t * stride;
  if (q_rank > 0 && blockIdx.y == 0) {
    float ss = 0.f;
    for (int j = threadIdx.x; j < q_rank; j += blockDim.x) ss = fmaf(row[j], row[j], ss);
    const float f = 1.0f / sqrtf(block_sum(ss, scratch) / (float)q_rank + eps);
    for (int j = threadIdx.x; j < q_rank; j += blockDim.x) Num<TC>::store(cq + (size_t)t * q_rank + j, row[j] * f * q_gain[j]);
  }
  if (kv_rank > 0 && blockIdx.y == gridDim.y - 1) {
    const int pos = tok_pos[t];
    const int page = block_table[(size_t)tok_seq[t] * bt_stride + pos / RB_PAGE];
    TC* dst = pages + ((size_t)page * RB_PAGE + (size_t)(pos % RB_PAGE)) * page_width;
    const float* src = row + kv_col;
    float ss = 0.f;
    for (int j = threadIdx.x; j < kv_rank; j += blockDim.x) ss = fmaf(src[j], src[j], ss);
    const float f = 1.0f / sqrtf(block_sum(ss, scratch) / (float)kv_rank + eps);
    for (int j = threadIdx.x; j < kv_rank; j += blockDim.x) Num<TC>::store(dst + j, src[j] * f * kv_gain[j]);
    // behind the latent: the row's `rot` numbers at rot_col rotated by the position (not normed), then zeros up to page_width
    if (page_width > kv_rank) {
      const int half = rot / 2;
      const float* rsrc = row + rot_col;
      const float* cr = cos_t + (size_t)pos * half;
      const float* sr = sin_t + (size_t)pos * half;
      TC* rdst = dst + kv_rank;
      for (int i = threadIdx.x; i < half; i += blockDim.x) {
        const int a = style == 0 ? 2 * i : i, b = style == 0 ? 2 * i + 1 : i + half;
        float y0, y1;
        rotate_pair(rsrc[a], rsrc[b], cr[i], sr[i], y0, y1);
        Num<TC>::store(rdst + a, y0);
        Num<TC>::store(rdst + b, y1);
      }
      for (int i = rot + threadIdx.x; i < page_width - kv_rank; i += blockDim.x) Num<TC>::store(rdst + i, 0.f);
    }
  }
}

extern "C" int rb_latent_norm_store(const float* proj, long long stride, int q_rank, const float* q_gain, void* cq,
                                    int kv_col, int kv_rank, const float* kv_gain, void* pages, int dtype,
                                    const int32_t* tok_pos, const int32_t* tok_seq, const int32_t* block_table,
                                    int bt_stride, float eps, int n_tokens, void* stream) {
  RB_RECORDED(rb_latent_norm_store(proj, stride, q_rank, q_gain, cq, kv_col, kv_rank, kv_gain, pages, dtype, tok_pos, tok_seq,
                                   block_table, bt_stride, eps, n_tokens, stream));
  RB_REQUIRE(n_tokens >= 0 && q_rank >= 0 && kv_rank >= 0 && kv_col >= 0, "rb_latent_norm_store: bad sizes");
  RB_REQUIRE(stride >= q_rank && stride >= (long long)kv_col + kv_rank, "rb_latent_norm_store: the row stride is too short");
  RB_REQUIRE(kv_rank == 0 || (pages && block_table), "rb_latent_norm_store: a latent needs cache pages");
  if (n_tokens == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == RB_F32)
    latent_norm_store_kernel<float><<<dim3(n_tokens, q_rank > 0 && kv_rank > 0 ? 2 : 1), 256, 0, s>>>(proj, (size_t)stride, q_rank, q_gain, (float*)cq, kv_col, kv_rank,
                                                             kv_gain, (float*)pages, kv_rank, tok_pos, tok_seq, block_table, bt_stride, eps);
  else if (dtype == RB_BF16)
    latent_norm_store_kernel<bf16_t><<<dim3(n_tokens, q_rank > 0 && kv_rank > 0 ? 2 : 1), 256, 0, s>>>(proj, (size_t)stride, q_rank, q_gain, (bf16_t*)cq, kv_col, kv_rank,
                                                              kv_gain, (bf16_t*)pages, kv_rank, tok_pos, tok_seq, block_table, bt_stride, eps);
  else
    RB_REQUIRE(false, "rb_latent_norm_store: unknown dtype %d", dtype);
  RB_LAUNCH_CHECK();
  return 0;
}

// The `rot` numbers at x_rot_col of head h of the tokens t0.., rotated by the tokens' positions, go to y at y_rot_col, and what lies
// behind them in the head of y becomes zero.
template <typename TX, typename TY>
__device__ __forceinline__ void heads_rotated_part(const TX* __restrict__ x, TY* __restrict__ y, int t0, int nt, int h, int n_heads,
                                                   size_t x_hs, size_t y_hs, int rot, int x_rot_col, int y_rot_col,
                                                   const float* __restrict__ cos_t, const float* __restrict__ sin_t, int style,
                                                   const int32_t* __restrict__ tok_pos) {
  const int half = rot / 2, tail = (int)y_hs - y_rot_col - rot, per = half + tail;
  for (int idx = threadIdx.x; idx < nt * per; idx += blockDim.x) {
    const int tt = idx / per, i = idx - tt * per;
    const TX* src = x + ((size_t)(t0 + tt) * n_heads + h) * x_hs + x_rot_col;
    TY* dst = y + ((size_t)(t0 + tt) * n_heads + h) * y_hs + y_rot_col;
    if (i < half) {
      const size_t at = (size_t)tok_pos[t0 + tt] * half + i;
      const int a = style == 0 ? 2 * i : i, b = style == 0 ? 2 * i + 1 : i + half;
      float y0, y1;
      rotate_pair(Num<TX>::load(src + a), Num<TX>::load(src + b), cos_t[at], sin_t[at], y0, y1);
      Num<TY>::store(dst + a, y0);
      Num<TY>::store(dst + b, y1);
    } else {
      Num<TY>::store(dst + rot + (i - half), 0.f);
    }
  }
}

// ---------------------------------------------------------------- a product per head
// y[t, h, n] = sum_k w[h, k, n] * x[t, h, k]: H small matrices, stored [H, K, N] (the output index runs fastest, so
// that neighbouring lanes read neighbouring weights).  A workgroup of four waves takes HL_TOKENS tokens and 64 output
// columns of one head: the tokens' inputs in LDS, a lane per column with one sum per token; the waves share the inner
// index (wave w takes k = w, w + 4, ...), sixteen weights in flight per lane (the scheduler is told not to move a load
// down to its use: it would trade the registers for a trip to memory per weight), and add up through LDS in a fixed order.
#define HL_TOKENS 16
#define HL_WAVES 4
template <typename TX, typename TW, typename TY>
__global__ __launch_bounds__(RB_WAVE * HL_WAVES) void heads_linear_kernel(const TX* __restrict__ x, const TW* __restrict__ w,
                                                                          TY* __restrict__ y, int n_tokens, int n_heads, int n, int k,
                                                                          size_t x_hs, size_t y_hs, const float* __restrict__ gate,
                                                                          size_t gate_stride, int rot, int x_rot_col, int y_rot_col,
                                                                          const float* __restrict__ cos_t,
                                                                          const float* __restrict__ sin_t, int style,
                                                                          const int32_t* __restrict__ tok_pos, int n_col_tiles) {
  extern __shared__ float xs[];                  // [HL_TOKENS][k], then [HL_WAVES - 1][HL_TOKENS][64] partial sums
  float* part = xs + HL_TOKENS * k;
  const int t0 = blockIdx.x * HL_TOKENS, h = blockIdx.y;
  const int lane = threadIdx.x & (RB_WAVE - 1), wave = threadIdx.x / RB_WAVE;
  const int nt = n_tokens - t0 < HL_TOKENS ? n_tokens - t0 : HL_TOKENS;
  if ((int)blockIdx.z == n_col_tiles) {
    // one more workgroup per (tokens, head)
    heads_rotated_part(x, y, t0, nt, h, n_heads, x_hs, y_hs, rot, x_rot_col, y_rot_col, cos_t, sin_t, style, tok_pos);
    return;
  }
  // the tokens' inputs, eight loads in flight per lane (a step of few tokens is a chain of trips to memory otherwise)
  for (int base = 0; base < HL_TOKENS * k; base += 8 * RB_WAVE * HL_WAVES) {
    float v[8];
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int idx = base + it * RB_WAVE * HL_WAVES + threadIdx.x;
      const int tt = idx / k, kk = idx - tt * k;
      v[it] = (idx < HL_TOKENS * k && tt < nt) ? Num<TX>::load(x + ((size_t)(t0 + tt) * n_heads + h) * x_hs + kk) : 0.f;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int idx = base + it * RB_WAVE * HL_WAVES + threadIdx.x;
      if (idx < HL_TOKENS * k) xs[idx] = v[it];
    }
  }
  __syncthreads();
  const int col = blockIdx.z * RB_WAVE + lane;
  const bool on = col < n;
  const TW* wh = w + (size_t)h * k * n + (on ? col : 0);
  float acc[HL_TOKENS];
#pragma unroll
  for (int tt = 0; tt < HL_TOKENS; ++tt) acc[tt] = 0.f;
  int kk = wave;
  for (; kk + 15 * HL_WAVES < k; kk += 16 * HL_WAVES) {
    float wv[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) wv[j] = Num<TW>::load(wh + (size_t)(kk + j * HL_WAVES) * n);
    __builtin_amdgcn_sched_barrier(0);          // all sixteen loads are issued before the first is waited for
#pragma unroll
    for (int j = 0; j < 16; ++j)
#pragma unroll
      for (int tt = 0; tt < HL_TOKENS; ++tt) acc[tt] = fmaf(wv[j], xs[tt * k + kk + j * HL_WAVES], acc[tt]);
  }
  for (; kk < k; kk += HL_WAVES) {
    const float wv = Num<TW>::load(wh + (size_t)kk * n);
#pragma unroll
    for (int tt = 0; tt < HL_TOKENS; ++tt) acc[tt] = fmaf(wv, xs[tt * k + kk], acc[tt]);
  }
  if (wave > 0) {
#pragma unroll
    for (int tt = 0; tt < HL_TOKENS; ++tt) part[((wave - 1) * HL_TOKENS + tt) * RB_WAVE + lane] = acc[tt];
  }
  __syncthreads();
  if (wave > 0 || !on) return;
#pragma unroll
  for (int tt = 0; tt < HL_TOKENS; ++tt) {
    float v = acc[tt];
#pragma unroll
    for (int ww = 0; ww < HL_WAVES - 1; ++ww) v += part[(ww * HL_TOKENS + tt) * RB_WAVE + lane];
    if (tt < nt) {
      if (gate) v *= 1.0f / (1.0f + expf(-gate[(size_t)(t0 + tt) * gate_stride + h]));      // a gate per head on the way out
      Num<TY>::store(y + ((size_t)(t0 + tt) * n_heads + h) * y_hs + col, v);
    }
  }
}

struct HeadsLinearMore {      // what rides in the same launch: a gate per head on the outputs, a rotated part beside them
  const float* gate = nullptr;
  size_t gate_stride = 0;
  int rot = 0, x_rot_col = 0, y_rot_col = 0, style = 0;
  const float* cos_t = nullptr;
  const float* sin_t = nullptr;
  const int32_t* tok_pos = nullptr;
  bool has_rot = false;
};
template <typename TX, typename TW, typename TY>
static void launch_heads_linear(const void* x, const void* w, void* y, int n_tokens, int n_heads, int n, int k, size_t x_hs,
                                size_t y_hs, hipStream_t s, const HeadsLinearMore& m = HeadsLinearMore()) {
  const int n_col_tiles = (n + RB_WAVE - 1) / RB_WAVE;
  dim3 grid((n_tokens + HL_TOKENS - 1) / HL_TOKENS, n_heads, n_col_tiles + (m.has_rot ? 1 : 0));
  const size_t lds = ((size_t)HL_TOKENS * k + (size_t)(HL_WAVES - 1) * HL_TOKENS * RB_WAVE) * sizeof(float);
  heads_linear_kernel<TX, TW, TY><<<grid, RB_WAVE * HL_WAVES, lds, s>>>((const TX*)x, (const TW*)w, (TY*)y, n_tokens, n_heads, n, k, x_hs,
                                                                        y_hs, m.gate, m.gate_stride, m.rot, m.x_rot_col, m.y_rot_col,
                                                                        m.cos_t, m.sin_t, m.style, m.tok_pos, n_col_tiles);
}

// The same products on the matrix cores: bfloat16 weights, fragment-major per head ([H][N / 16][K / 32] blocks of 1 KB, see
// gemm_internal.h), K a multiple of 32 up to 128, N of 16.  A wave takes 16 tokens of one head, holds their inputs as operands, and
// walks `tiles` of the head's blocks of 16 outputs, so that all of a wave's loads are on their way at once: the vector kernel above
// was a chain of three trips to memory in single-token steps, and a lane a column could not keep up with prompts.  Float32 inputs
// go in as three bfloat16 numbers each (the 24 bits of the significand cut in three, x = hi + mid + lo without a remainder), so that
// every product is exact and is summed in float32, as in the vector kernel.  Measured, 16 heads of 128 by 128:
// four tokens 9.7 -> 3.7 us from float32 and 4.5 from bfloat16, 3,782 tokens 82 -> 18 and 16; 32 heads of 64 by 96 with a rotated part,
// 3,782 tokens 93 -> 31.
template <typename TX>
struct HeadInput;
template <>
struct HeadInput<bf16_t> {
  static constexpr int PARTS = 1;
  static __device__ __forceinline__ void load(const bf16_t* p, Frag8 (&out)[1]) { out[0].u = load16(p); }
};
template <>
struct HeadInput<float> {
  static constexpr int PARTS = 3;
  static __device__ __forceinline__ void cut(float v, uint32_t (&part)[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      part[i] = __float_as_uint(v) >> 16;
      // an infinity or a NaN has no remainder
      v = (part[i] & 0x7f80u) == 0x7f80u ? 0.f : v - __uint_as_float(part[i] << 16);
    }
  }
  static __device__ __forceinline__ void load(const float* p, Frag8 (&out)[3]) {
    const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t w[3][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t lo[3], hi[3];
      cut(v[2 * i], lo);
      cut(v[2 * i + 1], hi);
#pragma unroll
      for (int q = 0; q < 3; ++q) w[q][i] = lo[q] | (hi[q] << 16);
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) out[q].u = make_uint4(w[q][0], w[q][1], w[q][2], w[q][3]);
  }
};

template <typename TX, typename TY, int KS>
__global__ __launch_bounds__(256) void heads_mfma_kernel(const TX* __restrict__ x, const bf16_t* __restrict__ w, TY* __restrict__ y,
                                                         int n_tokens, int n_heads, int n, size_t x_hs, size_t y_hs,
                                                         const float* __restrict__ gate, size_t gate_stride, int rot, int x_rot_col,
                                                         int y_rot_col, const float* __restrict__ cos_t, const float* __restrict__ sin_t,
                                                         int style, const int32_t* __restrict__ tok_pos, int tiles) {
  const int h = blockIdx.y;
  if (blockIdx.z == 1) {
    for (int t0 = blockIdx.x * 16; t0 < n_tokens; t0 += gridDim.x * 16)
      heads_rotated_part(x, y, t0, n_tokens - t0 < 16 ? n_tokens - t0 : 16, h, n_heads, x_hs, y_hs, rot, x_rot_col, y_rot_col, cos_t, sin_t,
                         style, tok_pos);
    return;
  }
  const int lane = threadIdx.x & (RB_WAVE - 1), r = lane & 15, kq = lane >> 4;
  const int id = blockIdx.x * (blockDim.x / RB_WAVE) + threadIdx.x / RB_WAVE;
  const int n_tiles = n / 16, groups = (n_tiles + tiles - 1) / tiles;
  const int t0 = id / groups * 16, first = id % groups * tiles;
  if (t0 >= n_tokens) return;
  const int last = first + tiles < n_tiles ? first + tiles : n_tiles;
  const bf16_t* wt = w + ((size_t)h * n_tiles + first) * (KS * 512) + 8 * lane;
  const int t = t0 + r < n_tokens ? t0 + r : n_tokens - 1;      // a token behind the last: the last one's numbers, never stored
  Frag8 a[KS], b[KS][HeadInput<TX>::PARTS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) a[ks].u = load16(wt + 512 * ks);
  const TX* xr = x + ((size_t)t * n_heads + h) * x_hs + 8 * kq;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) HeadInput<TX>::load(xr + 32 * ks, b[ks]);
  const float g = gate ? 1.0f / (1.0f + expf(-gate[(size_t)t * gate_stride + h])) : 1.0f;      // a gate per head on the way out
  TY* yr = y + ((size_t)t * n_heads + h) * y_hs + 4 * kq;
  for (int tile = first; tile < last; ++tile) {
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = HeadInput<TX>::PARTS - 1; q >= 0; --q)         // the smallest parts first
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) acc = mfma16(a[ks], b[ks][q], acc);
    if (tile + 1 < last) {
      wt += KS * 512;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) a[ks].u = load16(wt + 512 * ks);
    }
    acc *= g;
    if (t0 + r < n_tokens) {
      if constexpr (sizeof(TY) == 2)
        *reinterpret_cast<uint2*>(yr + 16 * tile) = make_uint2(pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3]));
      else
        *reinterpret_cast<f32x4_t*>(yr + 16 * tile) = acc;
    }
  }
}

template <typename TX, typename TY>
static void launch_heads_mfma(const void* x, const void* w, void* y, int n_tokens, int n_heads, int n, int k, size_t x_hs, size_t y_hs,
                              hipStream_t s, const HeadsLinearMore& m) {
  // single-token steps: a wave per 16 outputs; prompts: a wave per 16 tokens, while that gives every SIMD of the GPU a few
  const long long token_tiles = ((long long)n_tokens + 15) / 16, n_tiles = n / 16;
  int tiles = 1;
  while (tiles < n_tiles && token_tiles * n_heads * ((n_tiles + tiles - 1) / tiles) > 16LL * rb_compute_units()) tiles *= 2;
  const long long waves = token_tiles * ((n_tiles + tiles - 1) / tiles);
  const dim3 grid((unsigned)((waves + 3) / 4), n_heads, m.has_rot ? 2 : 1);
#define HM_GO(KS)                                                                                                                  \
  heads_mfma_kernel<TX, TY, KS><<<grid, 256, 0, s>>>((const TX*)x, (const bf16_t*)w, (TY*)y, n_tokens, n_heads, n, x_hs, y_hs, m.gate, \
                                                     m.gate_stride, m.rot, m.x_rot_col, m.y_rot_col, m.cos_t, m.sin_t, m.style,    \
                                                     m.tok_pos, tiles)
  if (k == 32) HM_GO(1);
  else if (k == 64) HM_GO(2);
  else if (k == 96) HM_GO(3);
  else HM_GO(4);
#undef HM_GO
}

// y[t, h, :n] = w[h]^T x[t, h, :k] (w [H, K, N]): a head of x takes x_head_stride numbers (the first k are read), a head of y
// y_head_stride (the first n are written).  Two things may ride in the launch.  gate (float32, rows gate_stride apart; null: none): head h's outputs of token t
// are multiplied by sigmoid(gate[t * gate_stride + h]).  rot >= 0 (rot < 0: none): the `rot` numbers at x_rot_col of every head
// of x, rotated by the token's position (cos, sin [positions, rot / 2]; style 0: 2i with 2i + 1, 1: i with i + rot / 2), go to
// y at y_rot_col, and what lies behind them in a head of y becomes zero.  w_layout 1: every head's [N, K] fragment-major (bfloat16, K 32,
// 64, 96 or 128, N a multiple of 16, x and y and their heads on 16-byte boundaries): the matrix cores' kernel.
extern "C" int rb_heads_linear_more(const void* x, int x_dtype, long long x_head_stride, const void* w, int w_dtype, int w_layout, void* y,
                                    int y_dtype, long long y_head_stride, int n_tokens, int n_heads, int n, int k, const float* gate,
                                    long long gate_stride, int rot, int x_rot_col, int y_rot_col, const float* cos, const float* sin,
                                    int style, const int32_t* tok_pos, void* stream) {
  RB_RECORDED(rb_heads_linear_more(x, x_dtype, x_head_stride, w, w_dtype, w_layout, y, y_dtype, y_head_stride, n_tokens, n_heads, n, k, gate,
                                   gate_stride, rot, x_rot_col, y_rot_col, cos, sin, style, tok_pos, stream));
  HeadsLinearMore more;
  more.gate = gate;
  more.gate_stride = (size_t)gate_stride;
  RB_REQUIRE(gate == nullptr || gate_stride >= n_heads, "rb_heads_linear: the gate's rows are shorter than the heads");
  if (rot >= 0) {
    RB_REQUIRE(rot % 2 == 0 && x_rot_col >= 0 && y_rot_col >= n && x_head_stride >= (long long)x_rot_col + rot &&
                   y_head_stride >= (long long)y_rot_col + rot,
               "rb_heads_linear: the rotated part lies outside a head, or over the product's outputs");
    RB_REQUIRE(rot == 0 || (cos && sin && tok_pos && (style == 0 || style == 1)), "rb_heads_linear: a rotation needs its tables");
    more.has_rot = y_head_stride > y_rot_col;
    more.rot = rot;
    more.x_rot_col = x_rot_col;
    more.y_rot_col = y_rot_col;
    more.style = style;
    more.cos_t = cos;
    more.sin_t = sin;
    more.tok_pos = tok_pos;
  }
  RB_REQUIRE(n_tokens >= 0 && n_heads > 0 && n_heads <= 65535 && n > 0 && n <= 65535 * 64 && k > 0, "rb_heads_linear: bad sizes");
  RB_REQUIRE(k <= 768, "rb_heads_linear: inner size %d not supported (at most 768)", k);
  RB_REQUIRE(x_head_stride >= k && y_head_stride >= n, "rb_heads_linear: a head's stride is shorter than the head");
  if (n_tokens == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const size_t xs = (size_t)x_head_stride, ys = (size_t)y_head_stride;
  if (w_layout == 1) {
    const long long x_size = x_dtype == RB_F32 ? 4 : 2, y_size = y_dtype == RB_F32 ? 4 : 2;
    RB_REQUIRE(w_dtype == RB_BF16 && k % 32 == 0 && k <= 128 && n % 16 == 0, "rb_heads_linear: fragment-major weights of %d x %d", n, k);
    RB_REQUIRE(((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(y)) & 15) == 0 &&
                   x_head_stride * x_size % 16 == 0 && y_head_stride * y_size % 16 == 0,
               "rb_heads_linear: the matrix cores' kernel needs heads on 16-byte boundaries");
    if (x_dtype == RB_F32 && y_dtype == RB_BF16) launch_heads_mfma<float, bf16_t>(x, w, y, n_tokens, n_heads, n, k, xs, ys, s, more);
    else if (x_dtype == RB_BF16 && y_dtype == RB_BF16) launch_heads_mfma<bf16_t, bf16_t>(x, w, y, n_tokens, n_heads, n, k, xs, ys, s, more);
    else RB_REQUIRE(false, "rb_heads_linear: this combination of types is not built fragment-major (x %d, y %d)", x_dtype, y_dtype);
    RB_LAUNCH_CHECK();
    return 0;
  }
  RB_REQUIRE(w_layout == 0, "rb_heads_linear: unknown layout %d", w_layout);
  const int key = x_dtype * 4 + w_dtype * 2 + y_dtype;
  switch (key) {
    case 0: launch_heads_linear<float, float, float>(x, w, y, n_tokens, n_heads, n, k, xs, ys, s, more); break;
    case 3: launch_heads_linear<float, bf16_t, bf16_t>(x, w, y, n_tokens, n_heads, n, k, xs, ys, s, more); break;
    case 6: launch_heads_linear<bf16_t, bf16_t, float>(x, w, y, n_tokens, n_heads, n, k, xs, ys, s, more); break;
    case 7: launch_heads_linear<bf16_t, bf16_t, bf16_t>(x, w, y, n_tokens, n_heads, n, k, xs, ys, s, more); break;
    case 2: launch_heads_linear<float, bf16_t, float>(x, w, y, n_tokens, n_heads, n, k, xs, ys, s, more); break;
    default: RB_REQUIRE(false, "rb_heads_linear: this combination of types is not built (x %d, w %d, y %d)", x_dtype, w_dtype, y_dtype);
  }
  RB_LAUNCH_CHECK();
  return 0;
}

// The product per head behind single-token attention whose splits are still to be put together (n_splits > 1; ws as rb_attention_decode_bf16_opts
// leaves it without an output, sinks as there): the result of a (sequence, head) goes to LDS as the bfloat16 numbers that attention would
// write, and through the head's matrix from there.  Bound by its trips to memory (maxima and sums, the splits, the weights beside them), as
// either launch was that it stands for; a workgroup a head, a wave 16 outputs.  Attention and product, us in a graph
// with the launch between them and without: 16 heads of 128 x 128, 1,500 keys in 16 splits, 1, 4 and 8 tokens 11.6 -> 9.8, 11.9 -> 10.2 and 12.2 ->
// 10.9; 12 and 16 tokens, which are two rounds of the workgroup's waves, 12.6 -> 12.9 and 12.8 -> 14.0.  So at most 8, where a wave has one row.
#define HC_THREADS 1024
#define HC_TOKENS 8
template <int D, int KS>
__global__ __launch_bounds__(HC_THREADS) void heads_combined_kernel(const float* __restrict__ ws, int n_splits, const float* __restrict__ sinks,
                                                                    const bf16_t* __restrict__ w, bf16_t* __restrict__ y, int n_tokens,
                                                                    int n_heads, int n, size_t y_hs, const float* __restrict__ gate,
                                                                    size_t gate_stride) {
  constexpr int LD = D + 8;                                // rows of the operand on different banks
  __shared__ __attribute__((aligned(16))) bf16_t xs[HC_TOKENS][LD];
  __shared__ float2 factors[HC_THREADS / RB_WAVE][RB_WAVE];
  const int h = blockIdx.x, lane = threadIdx.x & (RB_WAVE - 1), wave = threadIdx.x / RB_WAVE, r = lane & 15, kq = lane >> 4;
  const int n_tiles = n / 16;
  const bf16_t* wt = w + ((size_t)h * n_tiles + (wave < n_tiles ? wave : 0)) * (KS * 512) + 8 * lane;
  Frag8 a[KS], b[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) a[ks].u = load16(wt + 512 * ks);
  const int t = r < n_tokens ? r : n_tokens - 1;           // a token behind the last: the last one's numbers, never stored
  const float g = gate ? 1.0f / (1.0f + expf(-gate[(size_t)t * gate_stride + h])) : 1.0f;
  __builtin_amdgcn_sched_barrier(0);
  const int d = threadIdx.x % D;
  for (int row = threadIdx.x / D; row < n_tokens; row += HC_THREADS / D)
    xs[row][d] = f32_to_bf16(combined_split<D>(ws + ((size_t)row * n_heads + h) * n_splits * (D + 2), n_splits, sinks ? sinks + h : nullptr, false,
                                               factors[wave], lane, d));
  __syncthreads();
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) b[ks].u = *reinterpret_cast<const uint4*>(&xs[t][32 * ks + 8 * kq]);
  bf16_t* yr = y + ((size_t)t * n_heads + h) * y_hs + 4 * kq;
  for (int tile = wave; tile < n_tiles; tile += HC_THREADS / RB_WAVE) {
    if (tile != wave) {
      wt += (size_t)(HC_THREADS / RB_WAVE) * (KS * 512);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) a[ks].u = load16(wt + 512 * ks);
    }
    f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) acc = mfma16(a[ks], b[ks], acc);
    acc *= g;
    if (r < n_tokens) *reinterpret_cast<uint2*>(yr + 16 * tile) = make_uint2(pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3]));
  }
}

// Whether the kernel takes these sizes: latents of 64 or 128 numbers, of which the first k are read, and few tokens.
extern "C" int rb_heads_combined_ok(int n_tokens, int width, int n, int k) {
  return n_tokens >= 1 && n_tokens <= HC_TOKENS && (width == 64 || width == 128) && k > 0 && k % 32 == 0 && k <= width && n > 0 && n % 16 == 0;
}

// y[t, h, :n] = w[h]^T x[t, h, :k], x [T, H, width] the bfloat16 result of attention that lies as splits in ws; w fragment-major, y bfloat16, gate as in
// rb_heads_linear_more.
extern "C" int rb_heads_combined(const float* ws, int n_splits, const float* sinks, int width, const void* w, void* y, long long y_head_stride,
                                 int n_tokens, int n_heads, int n, int k, const float* gate, long long gate_stride, void* stream) {
  RB_RECORDED(rb_heads_combined(ws, n_splits, sinks, width, w, y, y_head_stride, n_tokens, n_heads, n, k, gate, gate_stride, stream));
  RB_REQUIRE(n_tokens == 0 || rb_heads_combined_ok(n_tokens, width, n, k), "rb_heads_combined: %d tokens, %d of %d numbers to %d are not for it",
             n_tokens, k, width, n);
  RB_REQUIRE(ws && w && y && n_splits > 1 && n_heads > 0 && n_heads <= 65535 && y_head_stride >= n && y_head_stride % 8 == 0,
             "rb_heads_combined: bad sizes");
  RB_REQUIRE(gate == nullptr || gate_stride >= n_heads, "rb_heads_combined: the gate's rows are shorter than the heads");
  RB_REQUIRE(((reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(y)) & 15) == 0, "rb_heads_combined: operands must be 16-byte aligned");
  if (n_tokens == 0) return 0;
#define HC_GO(D, KS)                                                                                                              \
  heads_combined_kernel<D, KS><<<n_heads, HC_THREADS, 0, (hipStream_t)stream>>>(ws, n_splits, sinks, (const bf16_t*)w, (bf16_t*)y, \
                                                                                n_tokens, n_heads, n, (size_t)y_head_stride, gate, \
                                                                                (size_t)gate_stride)
  if (width == 64) {
    if (k == 32) HC_GO(64, 1);
    else HC_GO(64, 2);
  } else {
    if (k == 32) HC_GO(128, 1);
    else if (k == 64) HC_GO(128, 2);
    else if (k == 96) HC_GO(128, 3);
    else HC_GO(128, 4);
  }
#undef HC_GO
  RB_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------- a rotated part beside the latent
// Where a head's key is a part made from the latent beside a rotated part that all heads share, the cache holds per token
// the latent c and, behind it, that rotated part: one key/value head of page_width >= kv_rank + rot numbers (the rest
// zeros), and a query is [Wk^T q_unrotated, rotate(q_rotated)] in the same layout.
// rb_latent_norm_store with that: the `rot` numbers at rot_col of a row of proj are rotated by the token's position
// (style 0: 2i with 2i + 1; 1: i with i + rot / 2; cos, sin [positions, rot / 2]) and stored behind the latent, by the same
// launch.
extern "C" int rb_latent_norm_rope_store(const float* proj, long long stride, int q_rank, const float* q_gain, void* cq, int kv_col,
                                         int kv_rank, const float* kv_gain, void* pages, int page_width, int rot_col, int rot,
                                         const float* cos, const float* sin, int style, int dtype, const int32_t* tok_pos,
                                         const int32_t* tok_seq, const int32_t* block_table, int bt_stride, float eps, int n_tokens,
                                         void* stream) {
  RB_RECORDED(rb_latent_norm_rope_store(proj, stride, q_rank, q_gain, cq, kv_col, kv_rank, kv_gain, pages, page_width, rot_col, rot,
                                        cos, sin, style, dtype, tok_pos, tok_seq, block_table, bt_stride, eps, n_tokens, stream));
  RB_REQUIRE(n_tokens >= 0 && q_rank >= 0 && kv_rank >= 0 && kv_col >= 0 && rot >= 0 && rot % 2 == 0 && rot_col >= 0,
             "rb_latent_norm_rope_store: bad sizes");
  RB_REQUIRE(stride >= q_rank && stride >= (long long)kv_col + kv_rank && stride >= (long long)rot_col + rot,
             "rb_latent_norm_rope_store: the row stride is too short");
  RB_REQUIRE(kv_rank == 0 || (pages && block_table && page_width >= kv_rank + rot),
             "rb_latent_norm_rope_store: a latent needs cache pages that hold it and the rotated part");
  RB_REQUIRE(rot == 0 || kv_rank == 0 || (cos && sin && (style == 0 || style == 1)), "rb_latent_norm_rope_store: a rotation needs its tables");
  RB_REQUIRE(dtype == RB_F32 || dtype == RB_BF16, "rb_latent_norm_rope_store: unknown dtype %d", dtype);
  if (n_tokens == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  if (dtype == RB_F32)
    latent_norm_store_kernel<float><<<dim3(n_tokens, q_rank > 0 && kv_rank > 0 ? 2 : 1), 256, 0, s>>>(proj, (size_t)stride, q_rank, q_gain, (float*)cq, kv_col, kv_rank,
                                                             kv_gain, (float*)pages, page_width, tok_pos, tok_seq, block_table,
                                                             bt_stride, eps, rot_col, rot, cos, sin, style);
  else
    latent_norm_store_kernel<bf16_t><<<dim3(n_tokens, q_rank > 0 && kv_rank > 0 ? 2 : 1), 256, 0, s>>>(proj, (size_t)stride, q_rank, q_gain, (bf16_t*)cq, kv_col, kv_rank,
                                                              kv_gain, (bf16_t*)pages, page_width, tok_pos, tok_seq, block_table,
                                                              bt_stride, eps, rot_col, rot, cos, sin, style);
  RB_LAUNCH_CHECK();
  return 0;
}
