// C[M, N] = A[M, K] * W[N, K]^T for any sizes, float32 or bfloat16 storage, float32
// multiply-add on the vector units or, for float32 operands with K % 16 == 0, the float32
// MFMA or, for many tokens, the bfloat16 MFMA on operands in three parts (gemm_f32.hip; never a reduced-precision matrix mode).  This is the
// whole float32 path's matrix product and the bfloat16 path's product for shapes the
// matrix-core kernels refuse.
//
// Reference: y[o] = sum_i W[i + o * n_in] * x[i] (llama/model.rs:67-91).
#include "api.h"
#include "common.h"
#include "gemm_internal.h"

#define GT 64      // tile of C: GT x GT
#define GK 16      // depth of one stage

template <typename TI, typename TO>
__global__ __launch_bounds__(256) void gemm_generic_kernel(const TI* __restrict__ a, const TI* __restrict__ w,
                                                           TO* __restrict__ c, int m, int n, int k) {
  __shared__ float as[GK][GT + 4];
  __shared__ float ws[GK][GT + 4];
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * GT;
  const int n0 = blockIdx.x * GT;
  const int tx = tid % 16;      // 4 columns of C each
  const int ty = tid / 16;      // 4 rows of C each
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

  // each thread loads 4 elements of the A tile and 4 of the W tile per stage
  const int lr = tid / 4;            // row of the tile, 0..63
  const int lk = (tid % 4) * 4;      // depth offset 0, 4, 8, 12
  for (int k0 = 0; k0 < k; k0 += GK) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int kk = k0 + lk + q;
      const int am = m0 + lr;
      const int wn = n0 + lr;
      as[lk + q][lr] = (am < m && kk < k) ? Num<TI>::load(a + (size_t)am * k + kk) : 0.f;
      ws[lk + q][lr] = (wn < n && kk < k) ? Num<TI>::load(w + (size_t)wn * k + kk) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < GK; ++kk) {
      float av[4], wv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) av[i] = as[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) wv[j] = ws[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int mm = m0 + ty * 4 + i;
    if (mm >= m) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int nn = n0 + tx * 4 + j;
      if (nn < n) Num<TO>::store(c + (size_t)mm * n + nn, acc[i][j]);
    }
  }
}

// Float32 operands and at most 16 tokens, depths that the two kernels below do not take: bound by reading W
// once.  A wave owns 4 rows of W and walks all of K with 16-byte loads (a row is read as
// 1 KB contiguous per instruction); the tokens' 1024-deep chunk goes through LDS once for
// the 4 waves; every lane keeps a partial sum per (row, token) and the wave adds them up at
// the end.  K must be a multiple of 4.
#define GS_ROWS 4
#define GS_KC 1024

template <int MT>
__global__ __launch_bounds__(256) void gemm_f32_skinny_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                              float* __restrict__ c, int m, int n, int k) {
  __shared__ float4 xs[MT][GS_KC / 4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int row0 = (blockIdx.x * 4 + wave) * GS_ROWS;
  float acc[GS_ROWS][MT];
#pragma unroll
  for (int r = 0; r < GS_ROWS; ++r)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[r][t] = 0.f;
  const float* wrow[GS_ROWS];
#pragma unroll
  for (int r = 0; r < GS_ROWS; ++r) wrow[r] = w + (size_t)(row0 + r < n ? row0 + r : n - 1) * k;

  for (int k0 = 0; k0 < k; k0 += GS_KC) {
    __syncthreads();                  // the previous chunk has been used by every wave
    for (int idx = tid; idx < MT * (GS_KC / 4); idx += 256) {
      const int t = idx / (GS_KC / 4), q = idx % (GS_KC / 4);
      const int kk = k0 + 4 * q;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (t < m && kk < k) v = *reinterpret_cast<const float4*>(a + (size_t)t * k + kk);
      xs[t][q] = v;
    }
    __syncthreads();
#pragma unroll
    for (int step = 0; step < GS_KC / 256; ++step) {
      const int q = step * 64 + lane;
      const int kk = k0 + 4 * q;
      const int kl = kk < k ? kk : k - 4;            // beyond K: a valid address; the tokens' chunk holds zeros there
      float4 wv[GS_ROWS];
#pragma unroll
      for (int r = 0; r < GS_ROWS; ++r) wv[r] = *reinterpret_cast<const float4*>(wrow[r] + kl);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const float4 xv = xs[t][q];
#pragma unroll
        for (int r = 0; r < GS_ROWS; ++r) {
          acc[r][t] = fmaf(wv[r].x, xv.x, acc[r][t]);
          acc[r][t] = fmaf(wv[r].y, xv.y, acc[r][t]);
          acc[r][t] = fmaf(wv[r].z, xv.z, acc[r][t]);
          acc[r][t] = fmaf(wv[r].w, xv.w, acc[r][t]);
        }
      }
    }
  }
#pragma unroll
  for (int r = 0; r < GS_ROWS; ++r)
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const float v = wave_sum(acc[r][t]);
      if (lane == 0 && row0 + r < n && t < m) c[(size_t)t * n + row0 + r] = v;
    }
}

// Float32 operands, at most 64 tokens, K a multiple of 128 (the float32 path's decode step at the
// widths of real models): bound by reading W once, and built like the bfloat16 product for few
// tokens.  The float32 MFMA 16x16x4 (float32 inputs, products and sums): rows of W are the
// matrix cores' row operand, the tokens their columns.  Lane l (row r = l % 16, group kq = l / 16)
// loads 16 bytes of row r at depth 16 j + 4 kq and feeds its four values to four MFMAs; the tokens
// are loaded the same way, so that an MFMA sums over the depths 16 j + 4 kq + i of its four groups
// (which depth a group holds is free as long as both operands agree).  A stage is 128 depth values:
// 8 loads of W per row tile, non-temporal (W is read once per step), all in flight while the stage
// before is multiplied.  K is dealt to the waves of a workgroup in stages and their partial sums
// meet in LDS in a fixed order.
typedef __attribute__((ext_vector_type(4))) float gf_f32x4_t;

// The gate's sums times those of the way up: which 0: the wave that has the gate's, 1: that has the others, -1: any other wave (all waves come here).
// silu as rb_swiglu computes it.
__device__ __forceinline__ gf_f32x4_t gated_end(gf_f32x4_t sum, float* __restrict__ lds, int lane, int which) {
  if (which == 1) *reinterpret_cast<gf_f32x4_t*>(lds + 4 * lane) = sum;
  __syncthreads();
  if (which != 0) return sum;
  const gf_f32x4_t u = *reinterpret_cast<const gf_f32x4_t*>(lds + 4 * lane);
#pragma unroll
  for (int i = 0; i < 4; ++i) sum[i] = sum[i] / (1.0f + expf(-sum[i])) * u[i];
  return sum;
}

// What stands before and after a product of at most 16 tokens in a step, done by the product (FOLD): the tokens are rows times a norm's gain, of which
// squares_in has the sums of squares over every 8 columns, and the sums are multiplied by the norm's factor; they are added to C and leave
// the same of C for the norm that follows.  Eight columns because a workgroup may have half of a tile's 16 rows.
// A norm of 4 rows as a launch of its own is 4 workgroups that wait twice for memory behind every product that ends a sublayer; what it leaves to the
// products is 384 sums of squares a token at width 3,072, asked for with the first stage, and one more number a lane to load and store.  Captured steps of
// 4 sequences, with such launches and so: width 3,072, 28 layers 3,126 and 3,049 us, width 96, 3 layers 124 and 122.
struct F32Fold {
  const float* squares_in;      // null: the tokens as they are; else [*, ceil(K / 8)]
  const int32_t* rows;          // which rows of x (and of squares_in) the tokens are; null: 0..M-1
  float eps;
  double per_k;                 // 1 / K
  int add;                      // C += the sums
  const float* gain;            // null: nothing for a norm; else [N], and
  float* gained;                //   [M, N] = C gain
  float* squares_out;           //   [M, ceil(N / 8)] = sums of C^2
  int wide;                     // C, the gain and the prepared rows can be read and written four columns at a time
};
constexpr int F32_SQ_WIDE = 8;
// A kernel that folds has one more argument.  The others have none: behind it the workgroup's size would no longer lie among the arguments that
// are there when a wave starts (28,672 rows at K = 4096, 22 tokens: 142.2 us with it, 140.5 without).
__device__ __forceinline__ F32Fold fold_of() { return F32Fold{}; }
__device__ __forceinline__ F32Fold fold_of(const F32Fold& fa) { return fa; }

__device__ __forceinline__ gf_f32x4_t four_of(const float* __restrict__ at, int left, int wide) {
  if (wide) return *reinterpret_cast<const gf_f32x4_t*>(at);
  gf_f32x4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (i < left) v[i] = at[i];
  return v;
}
__device__ __forceinline__ void put_four(float* __restrict__ at, gf_f32x4_t v, int left, int wide) {
  if (wide) {
    *reinterpret_cast<gf_f32x4_t*>(at) = v;
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (i < left) at[i] = v[i];
}
// The four lanes of a wave that share token r hold their shares of its squares: `lds` [waves][16] takes the waves' sums, before the barrier ...
__device__ __forceinline__ float squares_meet(float ss, float* __restrict__ lds, int wave, int lane) {
  ss += __shfl_xor(ss, 16, RB_WAVE);
  ss += __shfl_xor(ss, 32, RB_WAVE);
  if (lane < 16) lds[wave * 16 + lane] = ss;
  return ss;
}
// ... and behind it (with one wave there is none: its own sum) they make the norm's factor, in 64 bits.  The four roundings that it has in float32 (a mean,
// eps, a root, a quotient) meet all of a row's numbers alike: with them a model of width 96 was 2 % further off 64 bits than with norms in
// launches of their own (1.040e-7 for 1.021e-7), without them it is at 0.953e-7, in the same time.  One step from the root's estimate; infinity and 0,
// where the step is not a number, keep the estimate (0 and infinity).
__device__ __forceinline__ double squares_factor(float own, const float* __restrict__ lds, int n_waves, int lane, const F32Fold& fa) {
  float ss = own;
  if (n_waves > 1) {
    ss = 0.f;
    for (int ww = 0; ww < n_waves; ++ww) ss += lds[ww * 16 + (lane & 15)];
  }
  const double a = fma((double)ss, fa.per_k, (double)fa.eps), y = __builtin_amdgcn_rsq(a);
  return y > 0.0 && y < INFINITY ? y * fma(-0.5 * a * y, y, 1.5) : y;
}
__device__ __forceinline__ gf_f32x4_t times_factor(gf_f32x4_t sum, double factor) {
#pragma unroll
  for (int i = 0; i < 4; ++i) sum[i] = (float)((double)sum[i] * factor);
  return sum;
}
// The end of such a product: a lane's four sums of token mm, columns nn.. (both in range); lanes 16 apart have the two halves of 8 columns
__device__ __forceinline__ void fold_end(gf_f32x4_t v, gf_f32x4_t before, gf_f32x4_t gain, float* __restrict__ c, int mm, int nn, int n, bool in,
                                         int kq, const F32Fold& fa) {
  float sq = 0.f;
  if (in) {
    const int left = n - nn;
    if (fa.add) v += before;
    put_four(c + (size_t)mm * n + nn, v, left, fa.wide);
    if (fa.gain) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (i < left) sq = fmaf(v[i], v[i], sq);
      put_four(fa.gained + (size_t)mm * n + nn, v * gain, left, fa.wide);
    }
  }
  if (!fa.gain) return;
  sq += __shfl_xor(sq, 16, RB_WAVE);
  if (in && kq % 2 == 0) fa.squares_out[(size_t)mm * ((n + 7) / 8) + nn / 8] = sq;
}

// At most 16 tokens and a depth of at most 1,024 that is no multiple of 128 (K a multiple of 4, W as rows): a launch that is
// little more than its trips to memory.  Fragments as in the kernel below, a stage of 128 depth values per wave and trip, what lies
// behind K counts as zeros.  Every one of a stage's 32 products has an accumulator of its own, and they meet as a tree: no chain
// of dependent MFMAs, and an error like that of 64 lanes with a partial sum each (relative error at K = 96 / 500 / 1,000:
// 7.1e-8 / 8.4e-8 / 9.1e-8; the kernel above 7.1e-8 / 8.5e-8 / 9.9e-8; one accumulator for all of them 1.7e-7 / 2.0e-7 / 2.9e-7).
// 144 rows at K = 96, 4 / 16 tokens: 6.0 / 18.3 us in the kernel above, 3.0 / 3.1 here; 32,000 rows at K = 100 17.0 / 74.8 and 7.7 / 8.7.
// Its loads take 64 bytes of a row, the kernel above 1 KB: with many rows and K > 128 that one is the better for few tokens (32,000 rows
// at K = 500: 22.6 against 29.3 us with 4 tokens, 80 against 36 with 16; 4,096 rows at K = 1,000: 9.3 against 7.5).
// GATED: W is the gate's n rows and then n rows of the way up (n % 16 == 0), c [m, n] = silu(gate) up.  Twice the waves: the first half takes a tile of the
// gate, the other half the same rows of the way up, whose sums go to the first through LDS (gated_end).  The launch of 1 to 128 workgroups that
// did this behind the product cost a step 2 us; every sum and the gate are as they are in two launches.
template <bool GATED, typename... FOLDS>
__global__ __launch_bounds__(GATED ? 512 : 256) void gemm_f32_short_kernel(const float* __restrict__ x, const float* __restrict__ w, float* __restrict__ c,
                                                            int m, int n, int k, const FOLDS... folds) {
  constexpr bool FOLD = sizeof...(FOLDS) > 0;
  const F32Fold fa = fold_of(folds...);
  extern __shared__ float lds[];      // [waves - 1][4][64] for each of gate and way up, then, gated, [4][64], then, folded, [waves][16] for each
  const int lane = threadIdx.x & 63, n_waves = (blockDim.x >> 6) / (GATED ? 2 : 1);
  const int up = GATED && (int)(threadIdx.x >> 6) >= n_waves ? 1 : 0, wave = (threadIdx.x >> 6) - up * n_waves;
  float* red = lds + up * (n_waves - 1) * 256;
  const int r = lane & 15, kq = lane >> 4;
  const int n0 = blockIdx.x * 16;
  if (up) w += (size_t)n * k;
  // rows beyond N and tokens beyond M: row 0 and token 0, never stored
  const float* wrow = w + (size_t)(n0 + r < n ? n0 + r : 0) * k + 4 * kq;
  int from = r < m ? r : 0;
  if (FOLD && fa.rows) from = fa.rows[from];
  const float* xrow = x + (size_t)from * k + 4 * kq;
  const gf_f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  float* sq_lds = lds + (GATED ? 2 : 1) * (n_waves - 1) * 256 + (GATED ? 256 : 0) + up * n_waves * 16;
  SquaresShare<F32_SQ_WIDE> asked;
  gf_f32x4_t before = zero, gain = zero;
  const int nn = n0 + 4 * kq;
  const bool mine = r < m && nn < n;
  if (FOLD) {
    if (fa.squares_in) asked = squares_ask<F32_SQ_WIDE>(fa.squares_in + (size_t)from * ((k + 7) / 8), (k + 7) / 8, wave * 4 + kq, n_waves * 4);
    if (wave == 0 && mine && fa.add) before = four_of(c + (size_t)r * n + nn, n - nn, fa.wide);
    if (wave == 0 && mine && fa.gain) gain = four_of(fa.gain + nn, n - nn, fa.wide);
  }
  gf_f32x4_t acc[8][4];
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[j][i] = zero;
  for (int ks = 128 * wave; ks < k; ks += 128 * n_waves) {
    gf_f32x4_t a[8], b[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const bool in = ks + 16 * j + 4 * kq < k;
      a[j] = in ? *reinterpret_cast<const gf_f32x4_t*>(wrow + ks + 16 * j) : zero;
      b[j] = in ? *reinterpret_cast<const gf_f32x4_t*>(xrow + ks + 16 * j) : zero;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j][i], b[j][i], acc[j][i], 0, 0, 0);
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j][0] = (acc[j][0] + acc[j][1]) + (acc[j][2] + acc[j][3]);
  gf_f32x4_t sum = ((acc[0][0] + acc[1][0]) + (acc[2][0] + acc[3][0])) + ((acc[4][0] + acc[5][0]) + (acc[6][0] + acc[7][0]));
  float ss = 0.f;
  if (FOLD && fa.squares_in) ss = squares_meet(squares_sum(asked), sq_lds, wave, lane);
  if (n_waves > 1) {
    if (wave > 0)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[((wave - 1) * 4 + i) * 64 + lane] = sum[i];
    __syncthreads();
    if (!GATED && wave > 0) return;
    if (wave == 0)
      for (int o = 1; o < n_waves; ++o)
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] += red[((o - 1) * 4 + i) * 64 + lane];
  }
  if (FOLD && fa.squares_in && wave == 0) sum = times_factor(sum, squares_factor(ss, sq_lds, n_waves, lane, fa));
  if (GATED) {
    sum = gated_end(sum, lds + 2 * (n_waves - 1) * 256, lane, wave == 0 ? up : -1);
    if (wave > 0 || up) return;
  }
  if (FOLD && !GATED) {
    fold_end(sum, before, gain, c, r, nn, n, mine, kq, fa);
    return;
  }
  // lane l holds rows 4 (l / 16) + i of token l % 16
  if (r < m)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n0 + 4 * kq + i < n) c[(size_t)r * n + n0 + 4 * kq + i] = sum[i];
}

//
// At most 16 tokens, W fragment-major: XP blocks of 16 depth values that a load of the tokens brings, at most 16 / XP of them, and WP blocks
// that a load of W brings, a workgroup then having 16 / WP of the tile's rows (RowPack in gemm_internal.h; the same sums).  U: stages a wave has
// in registers.  A stage's 32 MFMAs add to one accumulator, 0.4 us one after the other, and behind them the next stage's loads took a trip to memory: with
// two sets of registers they are under way meanwhile.  Where workgroups share a compute unit they do that for each other, and a wave
// with more registers is slower (5,120 rows at K = 3072, 4 tokens: 14.9 us with one set, 15.9 with two).
// U = 0: one set as well, a stage's loads behind the multiplications of the one before, without FOLD in statements of its own: through the arrays and functions of the others, which say
// the same, the compiler asks for one load of W in front of the tokens, and 200 to 256 tiles of rows took 2 to 5 % more (4,096 rows at K = 4096, 16 tokens, 14.1 and 14.8 us); with
// barriers that fix the order of the loads 3 to 15 % more.  U = 1 keeps a block a load's tokens in front of W (4,096 rows at K = 4096, a workgroup
// a compute unit, 4 / 12 tokens: 12.5 / 13.4 us with U = 0, 14.7 / 14.8 with 1; 28,672 rows, 12 / 16 tokens: 89 / 96 and 78 / 88).
// GATED: as in the kernel above.
// FOLD: see F32Fold.
template <int MB, int R, bool WF, int XP = 1, int WP = 1, int U = 1, bool GATED = false, typename... FOLDS>
__global__ __launch_bounds__(GATED ? 512 : 256) void gemm_f32_few_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                          float* __restrict__ c, int m, int n, int k, const FOLDS... folds) {
  constexpr bool FOLD = sizeof...(FOLDS) > 0;
  const F32Fold fa = fold_of(folds...);
  extern __shared__ float lds[];      // [waves - 1][R * MB * 4][64] (for each of gate and way up, then [4][64]), then, folded, [waves][16] (for each)
  static_assert(!FOLD || (MB == 1 && R == 1), "folded: one tile of tokens and of rows");
  static_assert(!GATED || (MB == 1 && R == 1 && WP == 1), "gated: one tile of tokens, one of gate rows");
  constexpr int ACC = R * MB * 4;
  const int lane = threadIdx.x & 63, n_waves = (blockDim.x >> 6) / (GATED ? 2 : 1);
  const int up = GATED && (int)(threadIdx.x >> 6) >= n_waves ? 1 : 0, wave = (threadIdx.x >> 6) - up * n_waves;
  float* red = lds + up * (n_waves - 1) * ACC * 64;
  if (up) w += (size_t)n * k;
  const int r = lane & 15, kq = lane >> 4;
  static_assert((XP == 1 || MB == 1) && (WP == 1 || (MB == 1 && R == 1 && WF)), "packed operands: one tile of tokens");
  const int n0 = WP > 1 ? blockIdx.x / WP * 16 : blockIdx.x * (16 * R);
  const int part0 = WP > 1 ? blockIdx.x % WP * (16 / WP) : 0;      // WP > 1: this workgroup has 16 / WP of the tile's rows
  gf_f32x4_t acc[R][MB];
#pragma unroll
  for (int rt = 0; rt < R; ++rt)
#pragma unroll
    for (int cb = 0; cb < MB; ++cb) acc[rt][cb] = (gf_f32x4_t){0.f, 0.f, 0.f, 0.f};
  // Where a lane finds its 4 values at depth ks + 16 j + 4 kq of row tile rt: wrow[rt] + (ks + 16 j) * WK.
  // Rows [N, K]: the row's start + 4 kq, WK = 1.  Fragment-major (blocks of 16 rows x 16 depth values, 1 KB,
  // the 16 bytes of lane l at 16 l): the tile's start + 4 lane, WK = 16; a wave's load is then 1 KB in a
  // row, and W, read once per step, goes past the caches.
  constexpr int WK = WF ? 16 : 1;
  const float* wrow[R];
#pragma unroll
  for (int rt = 0; rt < R; ++rt) {
    const int row = n0 + 16 * rt + r;
    if (WP > 1) wrow[rt] = w + (size_t)n0 * k + 256 * (r / (16 / WP)) + 4 * (16 * kq + part0 + r % (16 / WP));
    else if (WF) wrow[rt] = w + (size_t)(n0 + 16 * rt < n ? n0 + 16 * rt : 0) * k + 4 * lane;
    else wrow[rt] = w + (size_t)(row < n ? row : 0) * k + 4 * kq;        // rows beyond N: row 0, never stored
  }
  const float* xrow[MB];
#pragma unroll
  for (int cb = 0; cb < MB; ++cb) {
    const int row = 16 * cb + r % (16 / XP);
    int from = row < m ? row : 0;
    if (FOLD && fa.rows) from = fa.rows[from];
    xrow[cb] = x + (size_t)from * k + 16 * (r / (16 / XP)) + 4 * kq;
  }
  float* sq_lds = lds + (GATED ? 2 : 1) * (n_waves - 1) * ACC * 64 + (GATED ? 256 : 0) + up * n_waves * 16;
  SquaresShare<F32_SQ_WIDE> asked;
  gf_f32x4_t before = {0.f, 0.f, 0.f, 0.f}, gain = before;
  const int nn_own = n0 + part0 + 4 * kq;
  const bool mine = r < m && nn_own < n && kq < 4 / WP;
  if (FOLD) {
    if (fa.squares_in) {
      int from = r < m ? r : 0;
      if (fa.rows) from = fa.rows[from];
      asked = squares_ask<F32_SQ_WIDE>(fa.squares_in + (size_t)from * ((k + 7) / 8), (k + 7) / 8, wave * 4 + kq, n_waves * 4);
    }
    if (wave == 0 && mine && fa.add) before = four_of(c + (size_t)r * n + nn_own, n - nn_own, fa.wide);
    if (wave == 0 && mine && fa.gain) gain = four_of(fa.gain + nn_own, n - nn_own, fa.wide);
  }
  // the K / 128 stages dealt to the waves as evenly as they go (the host launches no more waves than stages)
  const int total = k / 128, base = total / n_waves, extra = total % n_waves;
  const int stages = base + (wave < extra ? 1 : 0);
  const int k_begin = 128 * (wave * base + (wave < extra ? wave : extra));
  static_assert(U == 1 || (MB == 1 && R == 1 && WF), "no or two stages ahead: one tile of tokens and of rows, fragment-major");
  float ss = 0.f;
  if constexpr (U == 0 && !FOLD) {
    gf_f32x4_t a[R][8], b[MB][8];
    auto load_stage = [&](int st) {
      const int ks = k_begin + 128 * st;
#pragma unroll
      for (int j = 0; j < 8; ++j) a[0][j] = __builtin_nontemporal_load(reinterpret_cast<const gf_f32x4_t*>(wrow[0] + (size_t)(ks + 16 * j) * WK));
#pragma unroll
      for (int j = 0; j < 8; ++j) b[0][j] = *reinterpret_cast<const gf_f32x4_t*>(xrow[0] + ks + 16 * j);
    };
    auto multiply_stage = [&]() {
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[0][j][i], b[0][j][i], acc[0][0], 0, 0, 0);
    };
    load_stage(0);
    for (int st = 1; st < stages; ++st) {
      multiply_stage();
      load_stage(st);
    }
    multiply_stage();
  } else {
    gf_f32x4_t as[U == 2 ? 2 : 1][R][8 / WP], bs[U == 2 ? 2 : 1][MB][8 / XP];
    auto load_stage = [&](int u, int st) __attribute__((always_inline)) {
      auto &a = as[u];
      auto &b = bs[u];
      const int ks = k_begin + 128 * st;
      if constexpr (MB == 1 && U < 2 && XP == 1) {           // the tokens, which the caches hold, in front of W
#pragma unroll
        for (int j = 0; j < 8; ++j) b[0][j] = *reinterpret_cast<const gf_f32x4_t*>(xrow[0] + ks + 16 * j);
        if constexpr (U == 1) __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int j = 0; j < 8 / WP; ++j)
#pragma unroll
        for (int rt = 0; rt < R; ++rt)
          a[rt][j] = WF ? __builtin_nontemporal_load(reinterpret_cast<const gf_f32x4_t*>(wrow[rt] + (size_t)(ks + 16 * WP * j) * WK))
                        : *reinterpret_cast<const gf_f32x4_t*>(wrow[rt] + ks + 16 * WP * j);
      if constexpr (MB == 1 && U < 2 && XP == 1) return;
#pragma unroll
      for (int j = 0; j < 8 / XP; ++j)
#pragma unroll
        for (int cb = 0; cb < MB; ++cb) b[cb][j] = *reinterpret_cast<const gf_f32x4_t*>(xrow[cb] + ks + 16 * XP * j);
    };
    auto multiply_stage = [&](int u) __attribute__((always_inline)) {
      auto &a = as[u];
      auto &b = bs[u];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        gf_f32x4_t aj[R], bj[MB];
#pragma unroll
        for (int rt = 0; rt < R; ++rt) aj[rt] = RowPack<WP>::turned(a[rt][j / WP], j % WP);
#pragma unroll
        for (int cb = 0; cb < MB; ++cb) bj[cb] = RowPack<XP>::turned(b[cb][j / XP], j % XP);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int rt = 0; rt < R; ++rt)
#pragma unroll
            for (int cb = 0; cb < MB; ++cb) acc[rt][cb] = __builtin_amdgcn_mfma_f32_16x16x4f32(aj[rt][i], bj[cb][i], acc[rt][cb], 0, 0, 0);
      }
    };
    load_stage(0, 0);
    if (FOLD) {                          // the squares were asked for before the first stage and are added up before it arrives
      __builtin_amdgcn_sched_barrier(0);
      if (fa.squares_in) ss = squares_sum(asked);
    }
    if constexpr (U == 2) {
      int st = 0;
      for (; st + 2 < stages; st += 2) {
        load_stage(1, st + 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply_stage(0);
        load_stage(0, st + 2);
        __builtin_amdgcn_sched_barrier(0);
        multiply_stage(1);
      }
      if (st + 1 < stages) {
        load_stage(1, st + 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply_stage(0);
        multiply_stage(1);
      } else {
        multiply_stage(0);
      }
    } else {
      for (int st = 1; st < stages; ++st) {
        multiply_stage(0);
        load_stage(0, st);
      }
      multiply_stage(0);
    }
  }

  if (FOLD && fa.squares_in) ss = squares_meet(ss, sq_lds, wave, lane);
  if (n_waves > 1) {
    if (wave > 0) {
      float* dst = red + (size_t)(wave - 1) * ACC * 64 + lane;
#pragma unroll
      for (int rt = 0; rt < R; ++rt)
#pragma unroll
        for (int cb = 0; cb < MB; ++cb)
#pragma unroll
          for (int i = 0; i < 4; ++i) dst[((rt * MB + cb) * 4 + i) * 64] = acc[rt][cb][i];
    }
    __syncthreads();
    if (!GATED && wave != 0) return;
    for (int ww = 0; ww < (wave == 0 ? n_waves - 1 : 0); ++ww) {
      const float* src = red + (size_t)ww * ACC * 64 + lane;
#pragma unroll
      for (int rt = 0; rt < R; ++rt)
#pragma unroll
        for (int cb = 0; cb < MB; ++cb)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[rt][cb][i] += src[((rt * MB + cb) * 4 + i) * 64];
    }
  }
  if (FOLD && fa.squares_in && wave == 0) acc[0][0] = times_factor(acc[0][0], squares_factor(ss, sq_lds, n_waves, lane, fa));
  if constexpr (GATED) {
    acc[0][0] = gated_end(acc[0][0], lds + 2 * (n_waves - 1) * ACC * 64, lane, wave == 0 ? up : -1);
    if (wave > 0 || up) return;
  }
  // lane l holds, for token 16 cb + l % 16, the rows n0 + 16 rt + 4 (l / 16) + i
  if (WP > 1 && kq >= 4 / WP) return;
  if (FOLD && !GATED) {
    fold_end(acc[0][0], before, gain, c, r, nn_own, n, mine, kq, fa);
    return;
  }
#pragma unroll
  for (int rt = 0; rt < R; ++rt)
#pragma unroll
    for (int cb = 0; cb < MB; ++cb) {
      const int mm = 16 * cb + r, nn = n0 + part0 + 16 * rt + 4 * kq;
      if (mm >= m) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (nn + i < n) c[(size_t)mm * n + nn + i] = acc[rt][cb][i];
    }
}

static int g_f32_few = 1;
// experiments only: 0 = the float32 product of few tokens (W as rows) on the vector units; 3 = one row tile a wave whatever the sizes
extern "C" void rb_tune_f32_few(int on) { g_f32_few = on; }

static int g_f32_parts = 0;
extern "C" void rb_tune_f32_parts(int parts) { g_f32_parts = parts; }      // experiments and tests only: 1 or 2 workgroups for a tile of 16 rows; 0 = the built-in choice

// One row tile per wave and at most 4 waves: measured at 1 to 16 tokens on the products of the 8B shape with W
// fragment-major, two row tiles a wave lose everywhere but in the output matrix at 16 tokens (28,672 rows at
// K = 4096, 8 tokens: 78 us against 93; 4,096 rows at K = 14336: 38 against 54), and 4 waves are as fast as 8
// or faster (4,096 rows at K = 4096: 13.2 us against 14.4).  The kernel is never launched with more.
static int f32_few_waves(int k) { return k < 512 ? 1 : k < 1024 ? k / 256 : 4; }
// K = 96 of a step's few tokens and the like: see gemm_f32_short_kernel
static int f32_short_waves(int k) { return k <= 128 ? 1 : k <= 256 ? 2 : k <= 384 ? 3 : 4; }
static bool f32_short_takes(int m, int n, int k) {
  return m <= 16 && k % 4 == 0 && k <= 1024 && (k <= 128 || m > 8 || (long long)n * k <= 1 << 22) && g_f32_few;
}

// Whether a second stage under way pays where every tile has a workgroup (fragment-major W, at most a tile a compute unit): up to three tiles for four units and 12
// tokens, up to seven for eight and 8 tokens.  us without and with, of 256 units: 176 tiles, K = 4096, 4 / 8 / 12 / 13 tokens 11.5 / 12.0 / 12.5 / 12.6 and 10.3 / 11.3 / 12.5 / 12.9;
// 200 tiles 11.7 / 12.0 / 12.7 and 10.9 / 11.7 / 12.8; 224 11.8 / 12.3 / 12.7 and 11.6 / 12.1 / 13.4, K = 8192 22.3 / 22.9 / 23.4 and 21.2 / 22.2 / 24.1; 240 12.1 / 12.4 and 12.2 / 12.4; 256
// 12.6 / 12.7 and 13.1 / 13.1.
static bool f32_few_ahead(int m, int n) {
  const long long tiles = (n + 15) / 16, cus = rb_compute_units();
  return m <= 8 ? 8 * tiles <= 7 * cus : m <= 12 && 4 * tiles <= 3 * cus;
}
extern "C" int rb_tune_f32_ahead(int m, int n) { return f32_few_ahead(m, n); }      // for tests: the choice

// At most 16 tokens: one tile of them
template <typename... FOLDS>
static void launch_f32_16(const float* x, const float* w, bool w_frag, float* c, int m, int n, int k, hipStream_t s, const FOLDS&... folds) {
  constexpr bool FOLD = sizeof...(FOLDS) > 0;
  const int n_waves = f32_few_waves(k), grid = (n + 15) / 16;
  const size_t lds = ((size_t)(n_waves - 1) * 256 + (FOLD ? n_waves * 16 : 0)) * sizeof(float);
  // us, 4 tokens, as the kernel was (one stage, a block a load, whole tiles) and so: 3,072 rows at K = 3072 9.75 and 8.8, at 8192 24.3 and 21.3; 2,048 at 2048
  // 7.2 and 5.9, 1,024 at 4096 10.8 and 8.3 (halves of tiles); more workgroups than compute units: 5,120 at 3072 17.4 and 14.9, 16,384 38.0 and 35.0,
  // 128,256 260 and 239, 6,144 at 4096 23.4 and 20.7.  Halves of more tiles than half the units lose (3,072 rows at 3072 11.9).
  if (w_frag) {
    const bool ahead = f32_few_ahead(m, n);
    const int cus = rb_compute_units(), parts = g_f32_parts ? g_f32_parts : 2 * grid <= cus ? 2 : 1, pack = m <= 4 ? 4 : m <= 8 ? 2 : 1;
    auto by = [&](auto four, auto two, auto one) { return pack == 4 ? four : pack == 2 ? two : one; };
    (parts == 2    ? by(gemm_f32_few_kernel<1, 1, true, 4, 2, 2, false, FOLDS...>, gemm_f32_few_kernel<1, 1, true, 2, 2, 2, false, FOLDS...>,
                        gemm_f32_few_kernel<1, 1, true, 1, 2, 2, false, FOLDS...>)
     : ahead       ? gemm_f32_few_kernel<1, 1, true, 1, 1, 2, false, FOLDS...>
     : grid <= cus ? gemm_f32_few_kernel<1, 1, true, 1, 1, 0, false, FOLDS...>      // (packed tokens: 4,096 rows at K = 4096 14.2 for 13.9)
                   : by(gemm_f32_few_kernel<1, 1, true, 4, 1, 1, false, FOLDS...>, gemm_f32_few_kernel<1, 1, true, 2, 1, 1, false, FOLDS...>,
                        gemm_f32_few_kernel<1, 1, true, 1, 1, 1, false, FOLDS...>))<<<parts * grid, 64 * n_waves, lds, s>>>(x, w, c, m, n, k, folds...);
    return;
  }
  gemm_f32_few_kernel<1, 1, false, 1, 1, 1, false, FOLDS...><<<grid, 64 * n_waves, lds, s>>>(x, w, c, m, n, k, folds...);
}

template <typename... FOLDS>
static void launch_f32_short(const float* x, const float* w, float* c, int m, int n, int k, hipStream_t s, const FOLDS&... folds) {
  constexpr bool FOLD = sizeof...(FOLDS) > 0;
  const int n_waves = f32_short_waves(k);
  const size_t lds = ((size_t)(n_waves - 1) * 256 + (FOLD ? n_waves * 16 : 0)) * sizeof(float);
  gemm_f32_short_kernel<false, FOLDS...><<<(n + 15) / 16, 64 * n_waves, lds, s>>>(x, w, c, m, n, k, folds...);
}

// gate and way up, and the gate (rb_gemm_f32_gated_ok)
template <typename... FOLDS>
static void launch_f32_gated(const float* x, const float* w, bool w_frag, float* c, int m, int ff, int k, hipStream_t s, const FOLDS&... folds) {
  constexpr bool FOLD = sizeof...(FOLDS) > 0;
  const int grid = ff / 16, n_waves = w_frag ? f32_few_waves(k) : f32_short_waves(k);
  const size_t lds = ((size_t)2 * (n_waves - 1) * 256 + 256 + (FOLD ? 2 * n_waves * 16 : 0)) * sizeof(float);
  auto kern = !w_frag                          ? gemm_f32_short_kernel<true, FOLDS...>
              : 2 * grid <= rb_compute_units() ? gemm_f32_few_kernel<1, 1, true, 1, 1, 2, true, FOLDS...>      // (8 waves a workgroup: as two workgroups above)
              : m <= 4                         ? gemm_f32_few_kernel<1, 1, true, 4, 1, 1, true, FOLDS...>
              : m <= 8                         ? gemm_f32_few_kernel<1, 1, true, 2, 1, 1, true, FOLDS...>
                                               : gemm_f32_few_kernel<1, 1, true, 1, 1, 1, true, FOLDS...>;
  kern<<<grid, 2 * 64 * n_waves, lds, s>>>(x, w, c, m, ff, k, folds...);
}

template <int MB>
static void launch_f32_few(const float* x, const float* w, bool w_frag, float* c, int m, int n, int k, hipStream_t s) {
  const int n_waves = f32_few_waves(k);
  // From 33 tokens on a wave reads three to four times as many bytes of tokens as of W for every stage: two row
  // tiles a wave halve that (28,672 rows at K = 4096 with 64 tokens: 220 us against 305; 128,256 rows: 868
  // against 1,335; with 33 tokens 227 against 262).
  if constexpr (MB >= 3) {
    // (such a wave holds 246 registers, so a compute unit runs one workgroup of them: only where that still
    // gives every compute unit two workgroups and more)
    if (g_f32_few != 3 && (n + 31) / 32 >= 2 * rb_compute_units()) {
      const size_t lds2 = (size_t)(n_waves - 1) * 2 * MB * 4 * 64 * sizeof(float);
      const int grid2 = (n + 31) / 32;
      if (w_frag) gemm_f32_few_kernel<MB, 2, true><<<grid2, 64 * n_waves, lds2, s>>>(x, w, c, m, n, k);
      else gemm_f32_few_kernel<MB, 2, false><<<grid2, 64 * n_waves, lds2, s>>>(x, w, c, m, n, k);
      return;
    }
  }
  const size_t lds = (size_t)(n_waves - 1) * MB * 4 * 64 * sizeof(float);
  const int grid = (n + 15) / 16;
  if (w_frag) gemm_f32_few_kernel<MB, 1, true><<<grid, 64 * n_waves, lds, s>>>(x, w, c, m, n, k);
  else gemm_f32_few_kernel<MB, 1, false><<<grid, 64 * n_waves, lds, s>>>(x, w, c, m, n, k);
}

// Float32 operands and more than 16 tokens with K a multiple of 16 that is not one of 32, or operands
// that are not 16-byte aligned (everything else: gemm_f32.hip): the float32 MFMA (v_mfma_f32_32x32x2_f32: float32 inputs, float32 products and
// sums; no reduced-precision mode).  128 x 128 tiles, 16 deep, one wave per 64 x 64 piece.  W
// and the tokens are read with 16-byte loads along K and stored in LDS depth-major
// ([k][row], rows padded by 4 floats), so that the 32 lanes that read one depth value of 32
// rows hit 32 different banks; the next tile's loads are in flight in registers while the
// current one is multiplied.  D layout of the MFMA: lane l holds column l % 32 (a token),
// rows 8 * (i / 4) + 4 * (l / 32) + i % 4 (rows of W).
typedef __attribute__((ext_vector_type(16))) float gf32x16_t;
#define GM_T 128
#define GM_K 16
#define GM_LD (GM_T + 4)

template <bool WF>
__global__ __launch_bounds__(256) void gemm_f32_mfma_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                            float* __restrict__ c, int m, int n, int k) {
  __shared__ float ws[2][GM_K][GM_LD];
  __shared__ float xs[2][GM_K][GM_LD];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n0 = blockIdx.x * GM_T, m0 = blockIdx.y * GM_T;
  const int wn0 = (wave & 1) * 64, wm0 = (wave >> 1) * 64;
  const int l32 = lane & 31, g = lane >> 5;

  gf32x16_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // staging: thread t loads, for q = t and t + 256, row q / 4 of the tile, depth values 4 (q % 4) .. + 3;
  // of a fragment-major W (blocks of 16 rows x 16 depth values, the 16 bytes of lane l at 16 l) the 16 bytes
  // q % 64 of the tile's block q / 64: row 16 (q / 64) + q % 16, depth values 4 ((q % 64) / 16) .. + 3
  const float* wp[2];
  const float* xp[2];
  int w_row[2], w_kk[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int q = tid + 256 * i;
    int xr = m0 + q / 4;
    if (xr > m - 1) xr = m - 1;            // rows beyond the matrix: a valid row, never stored
    xp[i] = x + (size_t)xr * k + 4 * (q % 4);
    if (WF) {
      int tile = n0 / 16 + q / 64;
      if (tile > n / 16 - 1) tile = n / 16 - 1;
      w_row[i] = 16 * (q / 64) + q % 16;
      w_kk[i] = 4 * ((q % 64) / 16);
      wp[i] = w + (size_t)tile * 16 * k + 4 * (q % 64);
    } else {
      int wr = n0 + q / 4;
      if (wr > n - 1) wr = n - 1;
      w_row[i] = q / 4;
      w_kk[i] = 4 * (q % 4);
      wp[i] = w + (size_t)wr * k + 4 * (q % 4);
    }
  }
  float4 wreg[2], xreg[2];
  auto load_tile = [&](int kt) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      wreg[i] = *reinterpret_cast<const float4*>(wp[i] + (size_t)kt * (WF ? 256 : GM_K));
      xreg[i] = *reinterpret_cast<const float4*>(xp[i] + (size_t)kt * GM_K);
    }
  };
  auto store_tile = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int q = tid + 256 * i;
      const int row = q / 4, kk = 4 * (q % 4);
      ws[buf][w_kk[i] + 0][w_row[i]] = wreg[i].x;
      ws[buf][w_kk[i] + 1][w_row[i]] = wreg[i].y;
      ws[buf][w_kk[i] + 2][w_row[i]] = wreg[i].z;
      ws[buf][w_kk[i] + 3][w_row[i]] = wreg[i].w;
      xs[buf][kk + 0][row] = xreg[i].x;
      xs[buf][kk + 1][row] = xreg[i].y;
      xs[buf][kk + 2][row] = xreg[i].z;
      xs[buf][kk + 3][row] = xreg[i].w;
    }
  };
  const int k_tiles = k / GM_K;
  load_tile(0);
  store_tile(0);
  __syncthreads();
  for (int kt = 0; kt < k_tiles; ++kt) {
    const int buf = kt & 1;
    if (kt + 1 < k_tiles) load_tile(kt + 1);
#pragma unroll
    for (int ks = 0; ks < GM_K / 2; ++ks) {
      float a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i] = ws[buf][2 * ks + g][wn0 + 32 * i + l32];
#pragma unroll
      for (int j = 0; j < 2; ++j) b[j] = xs[buf][2 * ks + g][wm0 + 32 * j + l32];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    if (kt + 1 < k_tiles) store_tile(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int mm = m0 + wm0 + 32 * j + l32;
      if (mm >= m) continue;
      float* dst = c + (size_t)mm * n;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int nn = n0 + wn0 + 32 * i + 8 * (e / 4) + 4 * g + (e % 4);
        if (nn < n) dst[nn] = acc[i][j][e];
      }
    }
}

// Whether gate and way up of ff units each go in one launch with the gate on their sums (float32, W [2 ff, K] the gate's rows and then the others):
// at most 16 tokens, sizes that a product of them alone takes on the two kernels for few tokens.
extern "C" int rb_gemm_f32_gated_ok(int m, int ff, int k, int w_layout) {
  if (m < 1 || m > 16 || ff < 16 || ff % 16 != 0 || ff > 1 << 26 || k < 4 || !g_f32_few) return 0;
  if (w_layout == 1) return k % 128 == 0;
  return w_layout == 0 && k % 128 != 0 && f32_short_takes(m, 2 * ff, k);
}

// Whether that is also faster than the product and the gate in a launch each.  A compute unit that has one of these workgroups more has two tiles of rows more,
// where the product alone deals tile by tile (and halves of tiles where there are few): the launch pays where no unit gets more rows for it.
// us in two launches and in one, 4 tokens: 4,096 units of width 4096 (a tile of 16 a compute unit) 25.3 and 23.7, 8,192 45.8 and 44.1; 1,024 and 2,048 units, on which half of
// the GPU is idle, 11.4 and 19.5, 14.8 and 20.3; 5,120 (1.25 tiles a unit) 32.9 and 36.0; 14,336 (3.5) with 16 tokens 93.3 and 100.
// Depths of up to 512 are one trip to memory either way and the launch is what counts (1,024 units of 512 5.6 and 4.6), up to 1024 it still is with up to
// 8 tokens and more than a tile a unit (6,144 units 12.4 and 11.2); rows (the kernel for short depths) go by the first half of the rule alone (2,048 units of 1000 9.3 and
// 9.7, 5,120 with 16 tokens 24.5 and 23.1).
extern "C" int rb_gemm_f32_gated_pays(int m, int ff, int k, int w_layout) {
  if (!rb_gemm_f32_gated_ok(m, ff, k, w_layout)) return 0;
  const long long tiles = ff / 16, cus = rb_compute_units();
  if (k <= 512) return 1;
  if (2 * tiles <= cus) return 0;
  if (w_layout == 0 || (k <= 1024 && m <= 8 && tiles > cus)) return 1;
  return 2 * ((tiles + cus - 1) / cus) == (2 * tiles + cus - 1) / cus;
}

extern "C" int rb_gemm_f32_gated(const float* a, const float* w, int w_layout, float* c, int m, int ff, int k, void* stream) {
  RB_RECORDED(rb_gemm_f32_gated(a, w, w_layout, c, m, ff, k, stream));
  RB_REQUIRE(m == 0 || rb_gemm_f32_gated_ok(m, ff, k, w_layout), "rb_gemm_f32_gated: M=%d ff=%d K=%d, layout %d are not for it", m, ff, k, w_layout);
  RB_REQUIRE(((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w)) & 15) == 0, "rb_gemm_f32_gated: operands must be 16-byte aligned");
  if (m == 0) return 0;
  launch_f32_gated(a, w, w_layout == 1, c, m, ff, k, (hipStream_t)stream);
  RB_LAUNCH_CHECK();
  return 0;
}

// Whether a product of 1..16 float32 tokens takes its neighbours along (epilogue as in rb_gemm_f32_few): the sizes of the two kernels for few tokens.
extern "C" int rb_gemm_f32_few_ok(int m, int n, int k, int w_layout, int epilogue) {
  if (m < 1 || m > 16 || n < 1 || k < 4 || epilogue < 0 || epilogue > 3 || !g_f32_few) return 0;
  if (epilogue == 1) return n % 2 == 0 && rb_gemm_f32_gated_ok(m, n / 2, k, w_layout);
  if (w_layout == 1) return n % 16 == 0 && k % 128 == 0;
  return w_layout == 0 && (k % 128 == 0 || f32_short_takes(m, n, k));
}

// Whether a norm of rows of `width` is better done by the products around it than by a launch of its own: every workgroup of a product behind it reads all the sums
// of squares, which at more than 8 tokens or 3,072 columns takes longer than the launch.  Captured steps with launches and without, 1 / 4 / 8 / 9 / 16 sequences: width
// 2,048, 16 layers, 1,316 / 1,294 / 1,318 / 1,447 / 1,577 and 1,309 / 1,278 / 1,289 / 1,425 / 1,558 us; 3,072, 12 layers, 1,393 / 1,411 / 1,474 / 1,641 / 1,783 and 1,362 / 1,380 / 1,461 / 1,649 / 1,805; 4,096, 8
// layers, two shapes, 1,421 / 1,432 / 1,463 / 1,580 / 1,743 and 1,432 / 1,418 / 1,454 / 1,628 / 1,784, 1,402 / 1,368 / 1,413 / 1,594 / 1,736 and 1,415 / 1,377 / 1,423 / 1,627 / 1,769; 5,120, 6
// layers, 1,594 / 1,559 / 1,724 / 1,921 / 2,122 and 1,596 / 1,571 / 1,762 / 2,036 / 2,261.
extern "C" int rb_gemm_f32_fold_pays(int m, int width) { return m >= 1 && m <= 16 && width <= (m <= 8 ? 3072 : 2048); }

extern "C" int rb_gemm_f32_few(const float* a, const float* squares_in, float eps, const int32_t* rows, const float* w, int w_layout, float* c,
                               int epilogue, const float* gain, float* gained, float* squares_out, int m, int n, int k, void* stream) {
  RB_RECORDED(rb_gemm_f32_few(a, squares_in, eps, rows, w, w_layout, c, epilogue, gain, gained, squares_out, m, n, k, stream));
  RB_REQUIRE(rb_gemm_f32_few_ok(m, n, k, w_layout, epilogue), "rb_gemm_f32_few: M=%d N=%d K=%d, layout %d, epilogue %d are not for it", m, n, k,
             w_layout, epilogue);
  RB_REQUIRE(((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(squares_in)) & 15) == 0,
             "rb_gemm_f32_few: operands must be 16-byte aligned");
  RB_REQUIRE(!squares_in || epilogue <= 1, "rb_gemm_f32_few: prepared rows go with epilogues 0 and 1, not %d", epilogue);
  RB_REQUIRE(epilogue != 3 || (gain && gained && squares_out), "rb_gemm_f32_few: epilogue 3 needs the gain and room for the prepared rows");
  if (epilogue != 3) gain = nullptr, gained = squares_out = nullptr;
  const uintptr_t all = reinterpret_cast<uintptr_t>(c) | reinterpret_cast<uintptr_t>(gain) | reinterpret_cast<uintptr_t>(gained);
  const F32Fold fa = {squares_in, rows, eps, 1.0 / k, epilogue >= 2 ? 1 : 0, gain, gained, squares_out, n % 4 == 0 && (all & 15) == 0 ? 1 : 0};
  hipStream_t s = (hipStream_t)stream;
  if (epilogue == 1) launch_f32_gated(a, w, w_layout == 1, c, m, n / 2, k, s, fa);
  else if (k % 128 == 0) launch_f32_16(a, w, w_layout == 1, c, m, n, k, s, fa);
  else launch_f32_short(a, w, c, m, n, k, s, fa);
  RB_LAUNCH_CHECK();
  return 0;
}

extern "C" int rb_gemm_generic(const void* a, const void* w, int w_layout, void* c, int dtype_in, int dtype_out, int m,
                               int n, int k, void* stream) {
  RB_RECORDED(rb_gemm_generic(a, w, w_layout, c, dtype_in, dtype_out, m, n, k, stream));
  RB_REQUIRE(m >= 0 && n > 0 && k > 0, "rb_gemm_generic: bad sizes M=%d N=%d K=%d", m, n, k);
  // a fragment-major W is float32 with N % 16 == 0 and K % 128 == 0: sizes that the two matrix-core kernels take
  RB_REQUIRE(w_layout == 0 || (w_layout == 1 && dtype_in == RB_F32 && dtype_out == RB_F32 && n % 16 == 0 && k % 128 == 0),
             "rb_gemm_generic: W layout %d with dtype %d, N=%d K=%d (fragment-major: float32, N %% 16 == 0, K %% 128 == 0)",
             w_layout, dtype_in, n, k);
  const bool w_frag = w_layout == 1;
  if (m == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  if (dtype_in == RB_F32 && dtype_out == RB_F32 && m <= 64 && k % 128 == 0 && (g_f32_few || w_frag)) {
    const float* af = (const float*)a;
    const float* wf = (const float*)w;
    const int mb = (m + 15) / 16;
    if (mb == 1) launch_f32_16(af, wf, w_frag, (float*)c, m, n, k, s);
    else if (mb == 2) launch_f32_few<2>(af, wf, w_frag, (float*)c, m, n, k, s);
    else launch_f32_few<4>(af, wf, w_frag, (float*)c, m, n, k, s);
    RB_LAUNCH_CHECK();
    return 0;
  }
  if (dtype_in == RB_F32 && dtype_out == RB_F32 && f32_short_takes(m, n, k)) {
    launch_f32_short((const float*)a, (const float*)w, (float*)c, m, n, k, s);
    RB_LAUNCH_CHECK();
    return 0;
  }
  if (dtype_in == RB_F32 && dtype_out == RB_F32 && m <= 16 && k % 4 == 0) {
    const unsigned blocks = (unsigned)((n + 4 * GS_ROWS - 1) / (4 * GS_ROWS));
    const float* af = (const float*)a;
    const float* wf = (const float*)w;
    if (m <= 4) gemm_f32_skinny_kernel<4><<<blocks, 256, 0, s>>>(af, wf, (float*)c, m, n, k);
    else if (m <= 8) gemm_f32_skinny_kernel<8><<<blocks, 256, 0, s>>>(af, wf, (float*)c, m, n, k);
    else gemm_f32_skinny_kernel<16><<<blocks, 256, 0, s>>>(af, wf, (float*)c, m, n, k);
    RB_LAUNCH_CHECK();
    return 0;
  }
  if (dtype_in == RB_F32 && dtype_out == RB_F32 && m > 16) {
    int rc = 0;
    if (gemm_f32_dma_try((const float*)a, (const float*)w, w_frag, (float*)c, m, n, k, s, &rc)) {
      if (rc) return rc;
      RB_LAUNCH_CHECK();
      return 0;
    }
  }
  if (dtype_in == RB_F32 && dtype_out == RB_F32 && m > 16 && k % GM_K == 0) {
    dim3 tiles((n + GM_T - 1) / GM_T, (m + GM_T - 1) / GM_T);
    RB_REQUIRE(tiles.y <= 65535, "rb_gemm_generic: M=%d too large for one launch", m);
    if (w_frag) gemm_f32_mfma_kernel<true><<<tiles, 256, 0, s>>>((const float*)a, (const float*)w, (float*)c, m, n, k);
    else gemm_f32_mfma_kernel<false><<<tiles, 256, 0, s>>>((const float*)a, (const float*)w, (float*)c, m, n, k);
    RB_LAUNCH_CHECK();
    return 0;
  }
  RB_REQUIRE(!w_frag, "rb_gemm_generic: internal: a fragment-major W reached the kernels for rows");
  dim3 grid((n + GT - 1) / GT, (m + GT - 1) / GT);
  RB_REQUIRE(grid.y <= 65535, "rb_gemm_generic: M=%d too large for one launch", m);
  if (dtype_in == RB_F32 && dtype_out == RB_F32)
    gemm_generic_kernel<float, float><<<grid, 256, 0, s>>>((const float*)a, (const float*)w, (float*)c, m, n, k);
  else if (dtype_in == RB_BF16 && dtype_out == RB_F32)
    gemm_generic_kernel<bf16_t, float><<<grid, 256, 0, s>>>((const bf16_t*)a, (const bf16_t*)w, (float*)c, m, n, k);
  else if (dtype_in == RB_BF16 && dtype_out == RB_BF16)
    gemm_generic_kernel<bf16_t, bf16_t><<<grid, 256, 0, s>>>((const bf16_t*)a, (const bf16_t*)w, (bf16_t*)c, m, n, k);
  else
    RB_REQUIRE(false, "rb_gemm_generic: unsupported dtypes in=%d out=%d", dtype_in, dtype_out);
  RB_LAUNCH_CHECK();
  return 0;
}
