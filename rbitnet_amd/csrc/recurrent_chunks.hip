// Steps of many tokens through a layer that carries a matrix S [key size, value size] per head, in chunks of 16 tokens on the float32
// matrix core: the delta rule, the plain rule, and the rule that reads before it writes (the modes of rb_recurrence_step), with what
// enters the recurrence (unit vectors, decays, beta) made on the way.  All numbers are float32.
//
// With G_t the product of a chunk's decays up to and with token t (per key channel), the state before token t's write is
// diag(G_t) S_0 + sum_{s < t} diag(G_t / G_s) k_s u_s^T, so that for a chunk
//     (I + diag(beta) tril(A, -1)) U = diag(beta) (V - K^ S_0),   A[t, s] = sum_i k_ti k_si G_ti / G_si,   K^_t = G_t k_t
//     O = Q^ S_0 + tril(B) U,                                     B[t, s] = sum_i q_ti k_si G_ti / G_si,   Q^_t = G_t q_t
//     S_16 = diag(G_16) S_0 + K-^T U,                             K-_s = (G_16 / G_s) k_s
// (the plain rule: U = V; reading before the write: G_{t-1} in Q^ and B, and the bonus on B's diagonal).  A ratio G_t / G_s is a product
// of the decays between, so nothing is divided and nothing overflows.  16 tokens: A and B are sums with a ratio of their own for every
// pair of tokens and channel, 136 pairs, on the vector units; everything else is products.
//   1. chunk_operands: a workgroup per (chunk, head), all of them at once: A, B, T = (I + diag(beta) tril(A, -1))^-1, and with it
//      W = T diag(beta) K^ and T diag(beta) V, so that U = T diag(beta) V - W S_0.
//   2. chunk_walk: per (sequence, head, 16 columns of S) four waves that hold dim / 4 rows each walk the chunks: W S_0 and Q^ S_0 in parts
//      that meet in LDS, one barrier a chunk, the next chunk's operands on their way meanwhile.
// Operands lie in the workspace as the matrix core's lanes want them (an accumulator is the next product's operand as it is).
//
// A product of matrices carries an infinity or a NaN of one token to the tokens before it in its chunk, which walking does not: a chunk that
// has one is marked, its operands are k, q, decays, v and beta themselves, and the walk takes its tokens one after another.
//
// Bound by the float32 MFMAs of the walk (100 of 32 cycles for 16 tokens and 16 columns of 128 rows) while the longest sequence lasts, and
// in steps of many sequences by the operands' own sums.  3,781 tokens of four sequences, 16 heads of 128 x 128, the longest 1,500 tokens:
// 98 + 157 us, walked 546 + 62 for the launch that made the inputs; where it pays and where not: Kernels.recurrence_chunks_pay.  No
// further from 64 bits than walking is: the products of the decays are taken in 64 bits, which leaves one rounding where the walk has
// one a token (300 tokens, 4 heads of 128 x 48: states 1.28e-7 off, walked 1.36e-7; without decay 1.8e-6 and 5.4e-6).
#include <math.h>

#include "api.h"
#include "common.h"
#include "mfma.h"

namespace {

constexpr int CT = 16;                       // tokens of a chunk
enum { DELTA = 0, PLAIN = 1, BONUS = 2 };

__device__ __forceinline__ float sigmoid_of(float v) { return 1.0f / (1.0f + expf(-v)); }
__device__ __forceinline__ float softplus_of(float v) { return v > 20.0f ? v : log1pf(expf(v)); }
__device__ __forceinline__ bool finite(float v) { return fabsf(v) < INFINITY; }
__device__ __forceinline__ f32x4_t mfma4(float a, float b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// the sum over the 16 lanes of a row, in every lane of it
__device__ __forceinline__ float row_sum(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));   // quad_perm [1,0,3,2]
  v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, true));   // quad_perm [2,3,0,1]
  v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x141, 0xF, 0xF, true));  // row_half_mirror
  v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x140, 0xF, 0xF, true));  // row_mirror
  return v;
}

// A chunk's operands for one head: [W | Q^ | K- transposed | T beta V | B | G_16 | mark].  W and Q^ in tiles of 16 channels,
// [dim / 16][channels / 4][token][channel % 4]; K- [dim][token]; T beta V [vdim / 16][tokens / 4][column][token % 4]; B [token][token].
struct Places {
  int w, q, k, u, b, g, mark, size;
};
__host__ __device__ __forceinline__ Places places(int dim, int vdim) {
  Places p;
  p.w = 0;
  p.q = CT * dim;
  p.k = 2 * CT * dim;
  p.u = 3 * CT * dim;
  p.b = p.u + CT * vdim;
  p.g = p.b + CT * CT;
  p.mark = p.g + dim;
  p.size = p.mark + 16;
  return p;
}

template <int DIM, int MODE>
__global__ __launch_bounds__(256, DIM == 128 ? 5 : 3) void chunk_operands_kernel(const RbRecurrenceStep a, const int32_t* __restrict__ cu_seqlens, int first_chunk,
                                                             int window, float* __restrict__ ws) {
  constexpr int LD = DIM + 4;
  __shared__ __attribute__((aligned(16))) float lk[CT][LD], lq[CT][LD], lg[CT][LD];
  __shared__ __attribute__((aligned(16))) float la[CT][CT + 4], lb[CT][CT + 4], lt[CT][CT + 4];
  __shared__ float lbeta[CT];
  const int b = blockIdx.z, h = blockIdx.y, c = first_chunk + blockIdx.x;
  const int row0 = cu_seqlens[b] + CT * c, n = cu_seqlens[b + 1] - row0;
  if (n <= 0) return;
  const int nt = n < CT ? n : CT;
  const int tid = threadIdx.x, lane = tid & (RB_WAVE - 1), wave = tid / RB_WAVE;
  const int kvh = h / (a.n_heads / a.n_kv_heads);
  const Places at = places(DIM, a.vdim);
  float* out = ws + ((size_t)(b * window + blockIdx.x) * a.n_heads + h) * at.size;
  const bool one = a.a_per_head != 0;

  // ---- the tokens: 16 lanes a token.  Tokens behind the last have k = q = v = beta = 0 and decay 1: they change nothing
  const int tt = tid / 16, part = tid % 16;
  const bool live = tt < nt;
  const size_t row = (size_t)(row0 + (live ? tt : 0));
  bool bad = false;
  {
    float4 kv[DIM / 64], qv[DIM / 64], gv[DIM / 64];
    float4 bias[DIM / 64];
    float a1 = 0.f, araw = 0.f;
    if (one) araw = a.a[row * a.a_stride + h] + (a.a_bias ? a.a_bias[h] : 0.f);
    if (a.decay == 0) a1 = expf(a.a_log[h]);
#pragma unroll
    for (int j = 0; j < DIM / 64; ++j) {
      const int i = 4 * part + 64 * j;
      kv[j] = *reinterpret_cast<const float4*>(a.k + row * a.k_stride + (size_t)kvh * DIM + i);
      qv[j] = *reinterpret_cast<const float4*>(a.q + row * a.q_stride + (size_t)kvh * DIM + i);
      gv[j] = make_float4(araw, araw, araw, araw);
      if (!one) {
        gv[j] = *reinterpret_cast<const float4*>(a.a + row * a.a_stride + (size_t)h * DIM + i);
        if (a.a_bias) {
          const float* at4 = a.a_bias + (size_t)h * DIM + i;
          bias[j] = make_float4(at4[0], at4[1], at4[2], at4[3]);
          gv[j] = make_float4(gv[j].x + bias[j].x, gv[j].y + bias[j].y, gv[j].z + bias[j].z, gv[j].w + bias[j].w);
        }
      }
    }
    float fk = 1.f, fq = a.q_scale;
    if (a.unit) {
      float sk = 0.f, sq = 0.f;
#pragma unroll
      for (int j = 0; j < DIM / 64; ++j) {
        sk += (kv[j].x * kv[j].x + kv[j].y * kv[j].y) + (kv[j].z * kv[j].z + kv[j].w * kv[j].w);
        sq += (qv[j].x * qv[j].x + qv[j].y * qv[j].y) + (qv[j].z * qv[j].z + qv[j].w * qv[j].w);
      }
      fk = 1.0f / sqrtf(row_sum(sk) + a.unit_eps);
      fq = a.q_scale / sqrtf(row_sum(sq) + a.unit_eps);
    }
    auto decayed = [&](float z) {
      return a.decay == 0 ? expf(-a1 * softplus_of(z)) : a.decay == 1 ? expf(-softplus_of(-z) / a.tau) : expf(-expf(z));
    };
    float g1 = one ? decayed(araw) : 0.f;
#pragma unroll
    for (int j = 0; j < DIM / 64; ++j) {
      const int i = 4 * part + 64 * j;
      float4 k4 = make_float4(kv[j].x * fk, kv[j].y * fk, kv[j].z * fk, kv[j].w * fk);
      float4 q4 = make_float4(qv[j].x * fq, qv[j].y * fq, qv[j].z * fq, qv[j].w * fq);
      float4 g4 = one ? make_float4(g1, g1, g1, g1) : make_float4(decayed(gv[j].x), decayed(gv[j].y), decayed(gv[j].z), decayed(gv[j].w));
      if (!live) {
        k4 = q4 = make_float4(0.f, 0.f, 0.f, 0.f);
        g4 = make_float4(1.f, 1.f, 1.f, 1.f);
      }
      bad = bad || !(finite(k4.x) && finite(k4.y) && finite(k4.z) && finite(k4.w) && finite(q4.x) && finite(q4.y) && finite(q4.z) &&
                     finite(q4.w) && finite(g4.x) && finite(g4.y) && finite(g4.z) && finite(g4.w));
      *reinterpret_cast<float4*>(&lk[tt][i]) = k4;
      *reinterpret_cast<float4*>(&lq[tt][i]) = q4;
      *reinterpret_cast<float4*>(&lg[tt][i]) = g4;
    }
    if (live)
      for (int i = part; i < a.vdim; i += 16) bad = bad || !finite(a.v[row * a.v_stride + (size_t)h * a.vdim + i]);
    if (MODE == DELTA && part == 0) {
      const float beta = live ? sigmoid_of(a.b[row * a.b_stride + h]) : 0.f;
      bad = bad || !finite(beta);
      lbeta[tt] = beta;
    }
  }
  const bool mark = __syncthreads_or(bad) != 0;
  if (tid == 0) out[at.mark] = mark ? 1.f : 0.f;
  // v as the walk wants it: token 4 (lane / 16) + i, column 16 block + lane % 16
  auto value = [&](int block, int i) {
    const int t = 4 * (lane / 16) + i;
    return t < nt ? a.v[(size_t)(row0 + t) * a.v_stride + (size_t)h * a.vdim + 16 * block + lane % 16] : 0.f;
  };
  // a row of channels in the order of W and Q^: lane's token lane % 16, channels 16 tile + 4 (lane / 16) .. + 3
  const int ltok = lane % 16, lch = 4 * (lane / 16);
  if (mark) {
    for (int tile = wave; tile < DIM / 16; tile += 4) {
      *reinterpret_cast<float4*>(out + at.w + tile * 256 + 4 * lane) = *reinterpret_cast<const float4*>(&lk[ltok][16 * tile + lch]);
      *reinterpret_cast<float4*>(out + at.q + tile * 256 + 4 * lane) = *reinterpret_cast<const float4*>(&lq[ltok][16 * tile + lch]);
    }
    for (int i = tid; i < DIM * CT; i += 256) out[at.k + i] = lg[i % CT][i / CT];
    for (int block = wave; block < a.vdim / 16; block += 4)
      *reinterpret_cast<f32x4_t*>(out + at.u + block * 256 + 4 * lane) = (f32x4_t){value(block, 0), value(block, 1), value(block, 2), value(block, 3)};
    if (MODE == DELTA && tid < CT) out[at.b + tid] = lbeta[tid];
    return;
  }

  // ---- A and B: 16 lanes a token s, each with 4 or 8 channels, the ratio carried from token to token behind s
  {
    const int s = tt;
    float sa[CT], sb[CT];
#pragma unroll
    for (int t = 0; t < CT; ++t) sa[t] = sb[t] = 0.f;
#pragma unroll 1                              // (unrolled, every token's rows are asked for at once, and registers spill: 420 us for 60)
    for (int j = 0; j < DIM / 64; ++j) {
      const int i = 4 * part + 64 * j;
      float4 r = *reinterpret_cast<const float4*>(&lk[s][i]), own = r;
      if (MODE == BONUS) {
        const float* u = a.bonus + (size_t)h * DIM + i;
        own = make_float4(u[0] * r.x, u[1] * r.y, u[2] * r.z, u[3] * r.w);
      }
#pragma unroll
      for (int t = 0; t < CT; ++t) {
        const float4 g = *reinterpret_cast<const float4*>(&lg[t][i]), q = *reinterpret_cast<const float4*>(&lq[t][i]);
        const bool behind = t > s;
        if (MODE == BONUS) {                                 // the read sees the state before this token's decay
          const float4 m = t == s ? own : r;
          sb[t] = fmaf(q.w, m.w, fmaf(q.z, m.z, fmaf(q.y, m.y, fmaf(q.x, m.x, sb[t]))));
        }
        r = make_float4(behind ? r.x * g.x : r.x, behind ? r.y * g.y : r.y, behind ? r.z * g.z : r.z, behind ? r.w * g.w : r.w);
        if (MODE != BONUS) sb[t] = fmaf(q.w, r.w, fmaf(q.z, r.z, fmaf(q.y, r.y, fmaf(q.x, r.x, sb[t]))));
        if (MODE == DELTA) {
          const float4 k = *reinterpret_cast<const float4*>(&lk[t][i]);
          sa[t] = fmaf(k.w, r.w, fmaf(k.z, r.z, fmaf(k.y, r.y, fmaf(k.x, r.x, sa[t]))));
        }
      }
    }
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      const float vb = row_sum(sb[t]), va = MODE == DELTA ? row_sum(sa[t]) : 0.f;
      if (part == t) {
        lb[t][s] = t >= s ? vb : 0.f;
        if (MODE == DELTA) la[t][s] = t > s ? va : 0.f;
      }
    }
  }
  __syncthreads();

  // ---- T diag(beta): a column a lane, row after row; meanwhile the other waves take the products of the decays
  if (MODE == DELTA && tid < CT) {
    // (in LDS and not in registers: a column and the rows of A in registers left three workgroups on a compute unit, 115 us for 98)
#pragma unroll
    for (int t = 0; t < CT; ++t) lt[t][tid] = 0.f;
#pragma unroll 1
    for (int t = 0; t < CT; ++t) {
      float part_sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < CT; s += 4) {
        const float4 r = *reinterpret_cast<const float4*>(&la[t][s]);      // (zeros from s = t on)
        part_sum[0] = fmaf(r.x, lt[s][tid], part_sum[0]);
        part_sum[1] = fmaf(r.y, lt[s + 1][tid], part_sum[1]);
        part_sum[2] = fmaf(r.z, lt[s + 2][tid], part_sum[2]);
        part_sum[3] = fmaf(r.w, lt[s + 3][tid], part_sum[3]);
      }
      const float sum = (part_sum[0] + part_sum[1]) + (part_sum[2] + part_sum[3]);
      lt[t][tid] = (t == tid ? lbeta[tid] : 0.f) - lbeta[t] * sum;
    }
  }
  if (tid >= 128 && tid - 128 < DIM) {
    const int ch = tid - 128;
    // (in 64 bits: the products are what the walk has a rounding for in every token, and here they would all be one number's)
    double g[CT], behind = 1.0, upto = 1.0;
    float kb[CT];
#pragma unroll
    for (int t = 0; t < CT; ++t) g[t] = (double)lg[t][ch];
#pragma unroll
    for (int t = CT - 1; t >= 0; --t) {
      kb[t] = (float)((double)lk[t][ch] * behind);
      behind *= g[t];
    }
    out[at.g + ch] = (float)behind;
#pragma unroll
    for (int t = 0; t < CT; t += 4) *reinterpret_cast<float4*>(out + at.k + ch * CT + t) = make_float4(kb[t], kb[t + 1], kb[t + 2], kb[t + 3]);
#pragma unroll
    for (int t = 0; t < CT; ++t) {
      if (MODE == BONUS) lg[t][ch] = (float)upto;            // G before this token's own decay
      upto *= g[t];
      if (MODE != BONUS) lg[t][ch] = (float)upto;
    }
  }
  if (tid >= 64 && tid < 128) {
    const int e = 4 * (tid - 64);
    *reinterpret_cast<float4*>(out + at.b + e) = *reinterpret_cast<const float4*>(&lb[e / CT][e % CT]);
  }
  __syncthreads();

  f32x4_t tb = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  if (MODE == DELTA) tb = *reinterpret_cast<const f32x4_t*>(&lt[ltok][lch]);
  for (int tile = wave; tile < DIM / 16; tile += 4) {
    const float4 g = *reinterpret_cast<const float4*>(&lg[ltok][16 * tile + lch]), q = *reinterpret_cast<const float4*>(&lq[ltok][16 * tile + lch]);
    *reinterpret_cast<float4*>(out + at.q + tile * 256 + 4 * lane) = make_float4(q.x * g.x, q.y * g.y, q.z * g.z, q.w * g.w);
    if (MODE == DELTA) {                                     // W^T = K^^T (T diag(beta))^T: channels 4 (lane / 16) + i of token lane % 16
      f32x4_t w = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) w = mfma4(lk[lch + i][16 * tile + ltok] * lg[lch + i][16 * tile + ltok], tb[i], w);
      *reinterpret_cast<f32x4_t*>(out + at.w + tile * 256 + 4 * lane) = w;
    }
  }
  for (int block = wave; block < a.vdim / 16; block += 4) {
    f32x4_t v = (f32x4_t){value(block, 0), value(block, 1), value(block, 2), value(block, 3)};
    if (MODE == DELTA) {
      f32x4_t u = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) u = mfma4(tb[i], v[i], u);
      v = u;
    }
    *reinterpret_cast<f32x4_t*>(out + at.u + block * 256 + 4 * lane) = v;
  }
}

template <int DIM, int MODE>
__global__ __launch_bounds__(256) void chunk_walk_kernel(const RbRecurrenceStep a, const int32_t* __restrict__ cu_seqlens, int first_chunk,
                                                         int window, const float* __restrict__ ws, float* __restrict__ o) {
  constexpr int TILES = DIM / 64;            // tiles of 16 channels a wave holds
  __shared__ __attribute__((aligned(16))) f32x4_t parts[2][2][4][RB_WAVE];      // [chunk parity][W S, Q S][wave][lane]
  const int b = blockIdx.x / a.n_heads, h = blockIdx.x % a.n_heads, block = blockIdx.y;
  const int lane = threadIdx.x & (RB_WAVE - 1), wave = threadIdx.x / RB_WAVE;
  const int begin = cu_seqlens[b], len = cu_seqlens[b + 1] - begin;
  int chunks = (len + CT - 1) / CT - first_chunk;
  if (chunks > window) chunks = window;
  if (chunks <= 0) return;
  const Places at = places(DIM, a.vdim);
  const size_t step = (size_t)a.n_heads * at.size;
  const float* ops = ws + ((size_t)b * window * a.n_heads + h) * at.size;
  const int col = 16 * block + lane % 16, ch0 = wave * (DIM / 4) + 4 * (lane / 16);      // tile i: channels ch0 + 16 i .. + 3
  const int tile0 = wave * TILES;
  float* S = a.state + (((size_t)a.slots[b] * a.n_heads + h) * a.vdim + col) * DIM;
  f32x4_t s[TILES];
#pragma unroll
  for (int i = 0; i < TILES; ++i) s[i] = *reinterpret_cast<const f32x4_t*>(S + ch0 + 16 * i);

  struct Operands {
    f32x4_t w[TILES], q[TILES], k[TILES], g[TILES], u, b;
  };
  auto fetch = [&](int c) __attribute__((always_inline)) {
    const float* p = ops + (size_t)c * step;
    Operands r;
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
      if (MODE == DELTA) r.w[i] = *reinterpret_cast<const f32x4_t*>(p + at.w + (tile0 + i) * 256 + 4 * lane);
      r.q[i] = *reinterpret_cast<const f32x4_t*>(p + at.q + (tile0 + i) * 256 + 4 * lane);
      r.k[i] = *reinterpret_cast<const f32x4_t*>(p + at.k + ((tile0 + i) * 16 + lane % 16) * CT + 4 * (lane / 16));
      r.g[i] = *reinterpret_cast<const f32x4_t*>(p + at.g + ch0 + 16 * i);
    }
    r.u = *reinterpret_cast<const f32x4_t*>(p + at.u + block * 256 + 4 * lane);
    r.b = *reinterpret_cast<const f32x4_t*>(p + at.b + (lane % 16) * CT + 4 * (lane / 16));
    return r;
  };
  const f32x4_t zero = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  // a chunk whose operands are there
  auto chunk = [&](int c, const Operands& r) __attribute__((always_inline)) {
    const int t0 = CT * (first_chunk + c), nt = c >= chunks ? 0 : len - t0 < CT ? len - t0 : CT;
    float* orow = o + ((size_t)(begin + t0) * a.n_heads + h) * a.vdim + col;
    // Sums in two accumulators for every 16 channels, and the chunk's own part of the state and of the outputs in sums of their own: each
    // addition that meets a large running sum rounds at its size.
    f32x4_t wsum[2 * TILES], qsum[2 * TILES];
#pragma unroll
    for (int i = 0; i < 2 * TILES; ++i) wsum[i] = qsum[i] = zero;
#pragma unroll
    for (int i = 0; i < TILES; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (MODE == DELTA) wsum[2 * i + e / 2] = mfma4(r.w[i][e], s[i][e], wsum[2 * i + e / 2]);
        qsum[2 * i + e / 2] = mfma4(r.q[i][e], s[i][e], qsum[2 * i + e / 2]);
      }
    auto tree = [](const f32x4_t* v) { return TILES == 2 ? (v[0] + v[1]) + (v[2 * TILES - 2] + v[2 * TILES - 1]) : v[0] + v[1]; };
    if (MODE == DELTA) parts[c & 1][0][wave][lane] = tree(wsum);
    parts[c & 1][1][wave][lane] = tree(qsum);
    __syncthreads();
    auto whole = [&](int which) {
      const f32x4_t(*p)[RB_WAVE] = parts[c & 1][which];
      return (p[0][lane] + p[1][lane]) + (p[2][lane] + p[3][lane]);
    };
    const f32x4_t u = MODE == DELTA ? r.u - whole(0) : r.u;
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
      f32x4_t add0 = zero, add1 = zero;
      add0 = mfma4(r.k[i][0], u[0], add0);
      add1 = mfma4(r.k[i][2], u[2], add1);
      add0 = mfma4(r.k[i][1], u[1], add0);
      add1 = mfma4(r.k[i][3], u[3], add1);
      const f32x4_t add = add0 + add1;
#pragma unroll
      for (int e = 0; e < 4; ++e) s[i][e] = nt > 0 ? fmaf(s[i][e], r.g[i][e], add[e]) : s[i][e];
    }
    if (wave == (c & 3)) {                                   // one wave after the other writes the outputs
      f32x4_t y0 = zero, y1 = zero;
      y0 = mfma4(r.b[0], u[0], y0);
      y1 = mfma4(r.b[2], u[2], y1);
      y0 = mfma4(r.b[1], u[1], y0);
      y1 = mfma4(r.b[3], u[3], y1);
      const f32x4_t y = whole(1) + (y0 + y1);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int t = 4 * (lane / 16) + e;
        if (t < nt) orow[(size_t)t * a.n_heads * a.vdim] = y[e];
      }
    }
  };
  // a chunk with a number that is not finite: token after token
  auto walk = [&](int c) {
    const int t0 = CT * (first_chunk + c), nt = len - t0 < CT ? len - t0 : CT;
    float* orow = o + ((size_t)(begin + t0) * a.n_heads + h) * a.vdim + col;
    const float* p = ops + (size_t)c * step;
    for (int t = 0; t < nt; ++t) {
      float kv = 0.f, dq = 0.f, kq = 0.f;
      f32x4_t k[TILES], d[TILES];
#pragma unroll
      for (int i = 0; i < TILES; ++i) {
        const int tile = (tile0 + i) * 256 + (lane / 16) * 64 + 4 * t;
        k[i] = *reinterpret_cast<const f32x4_t*>(p + at.w + tile);
        const f32x4_t q = *reinterpret_cast<const f32x4_t*>(p + at.q + tile);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int ch = ch0 + 16 * i + e;
          kq = fmaf(MODE == BONUS ? a.bonus[(size_t)h * DIM + ch] * k[i][e] : k[i][e], q[e], kq);
          if (MODE == BONUS) dq = fmaf(s[i][e], q[e], dq);
          d[i][e] = s[i][e] * p[at.k + ch * CT + t];
          if (MODE == DELTA) kv = fmaf(d[i][e], k[i][e], kv);
          if (MODE != BONUS) dq = fmaf(d[i][e], q[e], dq);
        }
      }
      f32x4_t mine = (f32x4_t){kv, dq, kq, 0.f};
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        mine[e] += __shfl_xor(mine[e], 16, RB_WAVE);
        mine[e] += __shfl_xor(mine[e], 32, RB_WAVE);
      }
      __syncthreads();                                     // (the parts of the token, or the chunk, before have been read)
      parts[0][0][wave][lane] = mine;
      __syncthreads();
      f32x4_t all = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < 4; ++w) all += parts[0][0][w][lane];
      const float v = p[at.u + block * 256 + ((t / 4) * 16 + lane % 16) * 4 + t % 4];
      const float u = MODE == DELTA ? p[at.b + t] * (v - all[0]) : v;
#pragma unroll
      for (int i = 0; i < TILES; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[i][e] = fmaf(k[i][e], u, d[i][e]);
      if (wave == 0 && lane < 16) orow[(size_t)t * a.n_heads * a.vdim] = fmaf(u, all[2], all[1]);
    }
    __syncthreads();
  };
  bool marked = false;
  for (int c = lane; c < chunks; c += RB_WAVE) marked = marked || ops[(size_t)c * step + at.mark] != 0.f;
  if (__ballot(marked) != 0) {
    for (int c = 0; c < chunks; ++c) {
      if (ops[(size_t)c * step + at.mark] != 0.f) walk(c);
      else chunk(c, fetch(c));
    }
  } else {
    // A chunk's operands are asked for two chunks ahead, into the registers of the chunk that was just done: three sets, the loop written
    // out for each (a copy of a set would wait for its loads), and always asked for, so that the waits can count; chunks behind the
    // last leave the state as it is.
    const int last = chunks - 1;
    Operands one = fetch(0), two = fetch(last < 1 ? last : 1), three = fetch(last < 2 ? last : 2);
#pragma clang loop unroll(disable)
    for (int c = 0; c < chunks; c += 3) {
      chunk(c, one);
      one = fetch(last < c + 3 ? last : c + 3);
      chunk(c + 1, two);
      two = fetch(last < c + 4 ? last : c + 4);
      chunk(c + 2, three);
      three = fetch(last < c + 5 ? last : c + 5);
    }
  }
#pragma unroll
  for (int i = 0; i < TILES; ++i) *reinterpret_cast<f32x4_t*>(S + ch0 + 16 * i) = s[i];
}

}  // namespace

// Whether these sizes go in chunks.
extern "C" int rb_recurrence_chunks_ok(int n_heads, int n_kv_heads, int dim, int vdim) {
  return n_heads > 0 && n_kv_heads > 0 && n_heads % n_kv_heads == 0 && n_heads <= 65535 && (dim == 64 || dim == 128) && vdim > 0 &&
         vdim % 16 == 0 && vdim / 16 <= 65535;
}

// Floats of workspace for a window of `chunks` chunks (of 16 tokens) of every sequence.
extern "C" long long rb_recurrence_chunks_floats(int n_seqs, int n_heads, int dim, int vdim, int chunks) {
  return (long long)n_seqs * chunks * n_heads * places(dim, vdim).size;
}

// A step of any number of tokens per sequence (sequence b: rows cu_seqlens[b] .. of slot slots[b]) through the recurrence of `args` (its q,
// k, v, a, b as they are BEFORE unit vectors, decays and beta; mode 0, 1 or 2; convolution, gate, norm and out are not looked at), its
// outputs [T, H, vdim] float32 to o.  `window` chunks of every sequence at a time, the longest sequence having `chunks`; ws as
// rb_recurrence_chunks_floats(.., window) says.
extern "C" int rb_recurrence_chunks(const RbRecurrenceStep* args, const int32_t* cu_seqlens, int n_seqs, int chunks, int window, float* ws,
                                    float* o, void* stream) {
  RB_REQUIRE(args != nullptr, "rb_recurrence_chunks: no arguments");
  const RbRecurrenceStep a = *args;
  RB_RECORDED(rb_recurrence_chunks(&a, cu_seqlens, n_seqs, chunks, window, ws, o, stream));
  RB_REQUIRE(n_seqs >= 0 && n_seqs <= 65535 && chunks >= 0 && window >= 1 && rb_recurrence_chunks_ok(a.n_heads, a.n_kv_heads, a.dim, a.vdim),
             "rb_recurrence_chunks: %d heads on %d of %d x %d are not for it", a.n_heads, a.n_kv_heads, a.dim, a.vdim);
  RB_REQUIRE(a.mode >= DELTA && a.mode <= BONUS, "rb_recurrence_chunks: mode %d", a.mode);
  RB_REQUIRE(a.q && a.k && a.v && a.a && a.state && a.slots && cu_seqlens && ws && o, "rb_recurrence_chunks: a tensor is missing");
  RB_REQUIRE(!a.a_per_head || a.decay == 0, "rb_recurrence_chunks: decays per head are made with A_log");
  RB_REQUIRE((a.decay == 0 && a.a_log) || (a.decay == 1 && a.tau > 0.f) || a.decay == 2, "rb_recurrence_chunks: decay %d lacks its constants", a.decay);
  RB_REQUIRE((a.mode != DELTA || a.b) && (a.mode != BONUS || a.bonus), "rb_recurrence_chunks: a mode lacks its tensor");
  auto quads = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  RB_REQUIRE(quads(a.q) && quads(a.k) && quads(a.state) && quads(ws) && a.q_stride % 4 == 0 && a.k_stride % 4 == 0 &&
                 (a.a_per_head || (quads(a.a) && a.a_stride % 4 == 0)),
             "rb_recurrence_chunks: rows that are not aligned to 16 bytes");
  if (n_seqs == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
#define RC_GO(DIM, MODE)                                                                                                                  \
  do {                                                                                                                                    \
    chunk_operands_kernel<DIM, MODE><<<dim3(now, a.n_heads, n_seqs), 256, 0, s>>>(a, cu_seqlens, first, window, ws);                      \
    chunk_walk_kernel<DIM, MODE><<<dim3(n_seqs * a.n_heads, a.vdim / 16), 256, 0, s>>>(a, cu_seqlens, first, window, ws, o);              \
  } while (0)
#define RC_MODE(DIM)                          \
  do {                                        \
    if (a.mode == DELTA) RC_GO(DIM, DELTA);   \
    else if (a.mode == PLAIN) RC_GO(DIM, PLAIN); \
    else RC_GO(DIM, BONUS);                   \
  } while (0)
  for (int first = 0; first < chunks; first += window) {
    const int now = chunks - first < window ? chunks - first : window;
    if (a.dim == 128) RC_MODE(128);
    else RC_MODE(64);
  }
#undef RC_MODE
#undef RC_GO
  RB_LAUNCH_CHECK();
  return 0;
}
