// Products with few tokens (decode): bound by reading W once.  A wave owns 16*R rows of W and
// a slice of K, streams them with 16-byte loads straight into MFMA operands (W rows are the
// row operand, the tokens the columns, so a lane ends up with 4 consecutive outputs of one
// token), and the waves of a workgroup add their partial sums through LDS (no atomics: the
// sum order is fixed).
//
// Epilogue 1 expects W with gate and up rows interleaved in blocks of 16 and writes
// silu(gate) * up (llama/model.rs:297-302 of the reference) instead of the two products.
//
// What stands between two products of a decode step is folded into them (1..16 tokens):
//  * epilogue 2 adds the product to the float32 C it finds, the residual sum of
//    llama/model.rs:292-294 and :304-306; every element is read and written by one lane.
//  * epilogue 3 does the same and prepares the RMS norm that follows (llama/model.rs:93-100,
//    y_i = x_i * w_i / sqrt(mean(x^2) + eps)): it also writes bf16(x_i * w_i) and, for every 16
//    columns, the sum of x_i^2.  Both need the new x_i only, which the lane has at hand.
//  * SCALED: the tokens are such prepared rows.  The waves add up the sums of squares (in a
//    fixed order) while the product runs and the row's factor 1 / sqrt(..) is applied to the
//    float32 sums at the end.
// With both, no kernel runs between the products, and no row is read more often than before.
//
// Reference loop: y[o] = sum_i W[i + o * n_in] * x[i]  (llama/model.rs:67-91).
#include "api.h"
#include "tune.h"
#include "gemm_internal.h"

struct FoldArgs {
  const float* squares_in;      // SCALED: [*, ceil(K / 16)]
  const int32_t* rows;          // which rows of x (and of squares_in) the tokens are; null: 0..M-1
  float eps;
  const float* gain;            // epilogue 3: [N]
  bf16_t* gained;               // epilogue 3: [M, N]
  float* squares_out;           // epilogue 3: [M, ceil(N / 16)]
  int wide;                     // C, the gain and the prepared rows can be read and written four columns at a time
  int w_frag;                   // W is stored fragment-major (see gemm_internal.h)
  const float* act;             // epilogue 0: xIELU's two numbers, applied to the sums before they are stored; null: none
};

// Epilogue 0 with xIELU, a kernel of its own: as a run-time choice its code lay in the way of every product (2,048 rows at K = 2048,
// 4 tokens: 4.8 us with it, 4.5 without).
constexpr int EPI_ACT = 4;

// What a lane does with its 4 consecutive sums of token mm, columns nn.. (epilogues 0, 2, 3).
// All 64 lanes come here together: the sums of squares go round the four lanes that share
// a token's 16 columns.
// MAY: four columns at a time where FoldArgs::wide says so.  The squares are added up with fused operations that are spelled out: left to
// the compiler, the wide and the narrow store contracted them differently, and what is stored must not depend on addresses.
template <int EPI, bool MAY, typename TO>
__device__ __forceinline__ void store_sums(TO* __restrict__ c, const f32x4_t& sums, const f32x4_t& before,
                                           const f32x4_t& gain, int mm, int nn, int m, int n, int tile, int kq,
                                           const FoldArgs& fa) {
  const bool row_ok = mm < m;
  float sq = 0.f;
  XieluPair xa = {0.f, 0.f};
  if (EPI == EPI_ACT) xa = xielu_pair(fa.act);
  if (MAY && row_ok && fa.wide) {
    if (nn < n) {
      f32x4_t v = EPI == 2 || EPI == 3 ? before + sums : sums;
      if (EPI == EPI_ACT) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = xielu_value(v[i], xa.ap, xa.an);
      }
      TO* dst = c + (size_t)mm * n + nn;
      if constexpr (sizeof(TO) == 2) *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
      else *reinterpret_cast<f32x4_t*>(dst) = v;
      if (EPI == 3) {
#pragma unroll
        for (int i = 0; i < 4; ++i) sq = fmaf(v[i], v[i], sq);
        const f32x4_t p = v * gain;
        *reinterpret_cast<uint2*>(fa.gained + (size_t)mm * n + nn) = make_uint2(pack_bf16x2(p[0], p[1]), pack_bf16x2(p[2], p[3]));
      }
    }
  } else if (row_ok) {
    TO* dst = c + (size_t)mm * n + nn;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (nn + i >= n) continue;
      float v = EPI == 2 || EPI == 3 ? before[i] + sums[i] : sums[i];
      if (EPI == EPI_ACT) v = xielu_value(v, xa.ap, xa.an);
      Num<TO>::store(dst + i, v);
      if (EPI == 3) {
        sq = fmaf(v, v, sq);
        fa.gained[(size_t)mm * n + nn + i] = f32_to_bf16(v * gain[i]);
      }
    }
  }
  if (EPI == 3) {
    sq += __shfl_xor(sq, 16, RB_WAVE);
    sq += __shfl_xor(sq, 32, RB_WAVE);
    if (row_ok && kq == 0 && tile * 16 < n) fa.squares_out[(size_t)mm * ((n + 15) / 16) + tile] = sq;
  }
}

// FAST: K % 128 == 0, the K / 128 stages of 128 depth values dealt to the waves as evenly as they go, one stage in flight while the one
// before is multiplied; else any K % 8 == 0, with bounds checks.  WF (up to 16 tokens): W is stored fragment-major.
// (All of a wave's stages asked for at once instead, W's first, for up to four stages a wave: no faster at K = 128 to 4096 with any
// number of waves, 2,048 rows at K = 2048 4.5 us either way, 8,192 rows 7.6 -> 8.3.)
//
// XP: blocks of 32 depth values that a load of the tokens brings (see RowPack in gemm_internal.h).
// WP: blocks of depth that a load of W brings (one row tile a wave, W fragment-major): a workgroup then has 16 / WP of the tile's rows.
// ASIDE (a block a load): what was loaded is moved out of the way before it is multiplied, so that the next stage's W is asked for while the tokens of this
// one are waited for.  It costs registers, 2 to 48 a lane; see set_aside for who gains.
template <int MB, int R, bool FAST, bool WF, int EPI, typename TO, bool SCALED, int XP, int WP = 1, bool ASIDE = false>
__global__ __launch_bounds__(512) void gemm_skinny_kernel(const bf16_t* __restrict__ x,
                                                          const bf16_t* __restrict__ w, TO* __restrict__ c,
                                                          int m, int n, int k, int k_per_wave, FoldArgs fa) {
  // [waves - 1][R * MB][64] pieces of four sums, then, with SCALED, [waves - 1][MB][64] sums of squares
  extern __shared__ __attribute__((aligned(16))) float red[];
  constexpr int ACC = R * MB;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int n_waves = blockDim.x >> 6;
  const int r = lane & 15;
  const int kq = lane >> 4;
  static_assert(WP == 1 || (R == 1 && MB == 1 && FAST && WF && EPI != 1 && EPI != 3), "parts of a tile: one row tile a wave, ends that know no tile");
  const int n0 = WP > 1 ? blockIdx.x / WP * 16 : blockIdx.x * (16 * R);
  const int part0 = WP > 1 ? blockIdx.x % WP * (16 / WP) : 0;      // this workgroup's rows of the tile

  f32x4_t acc[R][MB];
#pragma unroll
  for (int rt = 0; rt < R; ++rt)
#pragma unroll
    for (int cb = 0; cb < MB; ++cb) acc[rt][cb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

  // Where a lane finds its 8 values at depth kstart (a multiple of 32) + 8 kq of row tile rt:
  // wrow[rt] + kstart * wk.  Rows [N, K]: the row's start + 8 kq, wk = 1.  Fragment-major: the
  // tile's start + 8 lane, wk = 16 (a block of 16 rows x 32 depth values is 512 values).
  const bool frag = MB == 1 ? WF : fa.w_frag != 0;      // (compiled in for up to 16 tokens)
  const int wk = frag ? 16 : 1;
  const bf16_t* wrow[R];
  bool wok[R];
#pragma unroll
  for (int rt = 0; rt < R; ++rt) {
    const int row = n0 + 16 * rt + r;
    wok[rt] = row < n;
    if (WP > 1) wrow[rt] = w + (size_t)n0 * k + 16 * RowPack<WP>::depth(r) + 8 * (16 * kq + part0 + RowPack<WP>::row(r));
    else if (frag) wrow[rt] = w + (size_t)(n0 + 16 * rt < n ? n0 + 16 * rt : 0) * k + 8 * lane;
    else wrow[rt] = w + (size_t)(wok[rt] ? row : 0) * k + 8 * kq;
  }
  static_assert(XP == 1 || (MB == 1 && FAST), "packed tokens: at most 8, whole stages");
  Frag8 a[R][4 / WP], b[MB][4 / XP];
  auto load_w = [&](int ks) {                         // depth values ks..ks + 127 of the wave's rows
#pragma unroll
    for (int j = 0; j < 4 / WP; ++j)
#pragma unroll
      for (int rt = 0; rt < R; ++rt) {
        const bf16_t* src = wrow[rt] + (size_t)(ks + 32 * WP * j) * wk;
        if (frag) a[rt][j].u = load16_stream(src);      // read once, whole lines at a time: past the caches
        else a[rt][j].u = load16(src);
      }
  };
  const bf16_t* xrow[MB];
  bool xok[MB];
  float ss[MB];
  SquaresShare<> asked[MB];
#pragma unroll
  for (int cb = 0; cb < MB; ++cb) {
    const int row = 16 * cb + r;
    xok[cb] = row < m;
    size_t src = xok[cb] ? row : 0;
    if (fa.rows) src = (size_t)fa.rows[src];
    xrow[cb] = x + src * k;
    if (XP > 1) {
      const int packed = RowPack<XP>::row(r) < m ? RowPack<XP>::row(r) : 0;
      xrow[cb] = x + (size_t)(fa.rows ? fa.rows[packed] : packed) * k + RowPack<XP>::depth(r);
    }
    ss[cb] = 0.f;
    if (SCALED) {
      const int n_sq = (k + 15) / 16;
      asked[cb] = squares_ask(fa.squares_in + src * n_sq, n_sq, wave * 4 + kq, n_waves * 4);
    }
  }

  // epilogues 2 and 3: what C holds now, and the gain, are asked for before the products, not
  // after them
  f32x4_t before[R][MB], gain[R];
#pragma unroll
  for (int rt = 0; rt < R; ++rt) {
    const int nn = n0 + part0 + 16 * rt + 4 * kq;
    gain[rt] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    if (EPI == 3 && wave == 0) {
      if (fa.wide) {
        if (nn < n) gain[rt] = *reinterpret_cast<const f32x4_t*>(fa.gain + nn);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (nn + i < n) gain[rt][i] = fa.gain[nn + i];
      }
    }
#pragma unroll
    for (int cb = 0; cb < MB; ++cb) {
      before[rt][cb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
      if ((EPI == 2 || EPI == 3) && wave == 0) {
        const int mm = 16 * cb + r;
        if (sizeof(TO) == 4 && fa.wide) {
          if (mm < m && nn < n) before[rt][cb] = *reinterpret_cast<const f32x4_t*>(c + (size_t)mm * n + nn);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (mm < m && nn + i < n) before[rt][cb][i] = Num<TO>::load(c + (size_t)mm * n + nn + i);
        }
      }
    }
  }

  auto multiply_stage = [&]() {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int rt = 0; rt < R; ++rt)
#pragma unroll
        for (int cb = 0; cb < MB; ++cb) {
          if constexpr (XP == 1 && WP == 1 && !ASIDE) acc[rt][cb] = mfma16(a[rt][j], b[cb][j], acc[rt][cb]);
          else acc[rt][cb] = mfma16(RowPack<WP>::block(a[rt], j), RowPack<XP>::block(b[cb], j), acc[rt][cb]);
        }
  };
  if constexpr (FAST) {
    // K and every wave's range are multiples of 128: no bounds checks.  Rows beyond N or M
    // are read from row 0 instead and their results never stored.
    // Every wave has at least one stage (the host launches no more waves than stages): the loads below are unconditional, which
    // lets the compiler count outstanding loads exactly.  The first K / 128 % waves waves take one stage more (K = 11008 = 86
    // stages over 8 waves: six times 11, twice 10).
    const int total = k / 128, base = total / n_waves, extra = total % n_waves;
    const int stages = base + (wave < extra ? 1 : 0);
    const int k_begin = 128 * (wave * base + (wave < extra ? wave : extra));
    auto load_stage = [&](int st) {
      const int ks = k_begin + 128 * st;
      load_w(ks);
#pragma unroll
      for (int j = 0; j < 4 / XP; ++j)
#pragma unroll
        for (int cb = 0; cb < MB; ++cb) b[cb][j].u = load16(xrow[cb] + ks + 8 * kq + 32 * XP * j);
    };
    load_stage(0);
    // the sums of squares were asked for before the first stage and arrive before it: added up
    // here, they do not occupy registers during the loop
    if (SCALED) {
#pragma unroll
      for (int cb = 0; cb < MB; ++cb) ss[cb] = squares_sum(asked[cb]);
    }
    for (int st = 1; st < stages; ++st) {
      multiply_stage();
      load_stage(st);
    }
    multiply_stage();
  } else {
    if (SCALED) {
#pragma unroll
      for (int cb = 0; cb < MB; ++cb) ss[cb] = squares_sum(asked[cb]);
    }
    const int k_begin = wave * k_per_wave, k_end = (k_begin + k_per_wave < k) ? k_begin + k_per_wave : k;
    for (int k0 = k_begin; k0 < k_end; k0 += 128) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int kk = k0 + 32 * j + 8 * kq;
        const bool in = kk < k_end;
#pragma unroll
        for (int rt = 0; rt < R; ++rt)
          a[rt][j / WP].u = (in && wok[rt]) ? load16(wrow[rt] + (size_t)(k0 + 32 * j) * wk) : zero16();
#pragma unroll
        for (int cb = 0; cb < MB; ++cb) b[cb][j / XP].u = (in && xok[cb]) ? load16(xrow[cb] + kk) : zero16();
      }
      multiply_stage();
    }
  }

  // ---- a token's squares: the four lanes that share its row add their shares
  if (SCALED) {
#pragma unroll
    for (int cb = 0; cb < MB; ++cb) {
      ss[cb] += __shfl_xor(ss[cb], 16, RB_WAVE);
      ss[cb] += __shfl_xor(ss[cb], 32, RB_WAVE);
    }
  }

  // ---- partial sums of waves 1.. go through LDS to wave 0
  if (n_waves > 1) {
    float* sq = red + (size_t)(n_waves - 1) * ACC * 256;
    if (wave > 0) {
      float* dst = red + (size_t)(wave - 1) * ACC * 256 + 4 * lane;
#pragma unroll
      for (int rt = 0; rt < R; ++rt)
#pragma unroll
        for (int cb = 0; cb < MB; ++cb) *reinterpret_cast<f32x4_t*>(dst + (rt * MB + cb) * 256) = acc[rt][cb];
      if (SCALED) {
#pragma unroll
        for (int cb = 0; cb < MB; ++cb) sq[((wave - 1) * MB + cb) * 64 + lane] = ss[cb];
      }
    }
    __syncthreads();
    if (wave == 0) {
      for (int ww = 0; ww < n_waves - 1; ++ww) {
        const float* src = red + (size_t)ww * ACC * 256 + 4 * lane;
#pragma unroll
        for (int rt = 0; rt < R; ++rt)
#pragma unroll
          for (int cb = 0; cb < MB; ++cb) acc[rt][cb] += *reinterpret_cast<const f32x4_t*>(src + (rt * MB + cb) * 256);
        if (SCALED) {
#pragma unroll
          for (int cb = 0; cb < MB; ++cb) ss[cb] += sq[(ww * MB + cb) * 64 + lane];
        }
      }
    }
  }
  if (wave != 0) return;

  if (SCALED) {
#pragma unroll
    for (int cb = 0; cb < MB; ++cb) {
      const float scale = 1.0f / sqrtf(ss[cb] / (float)k + fa.eps);
#pragma unroll
      for (int rt = 0; rt < R; ++rt)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[rt][cb][i] *= scale;
    }
  }

  // ---- lane holds, per (rt, cb): token 16*cb + r, W rows n0 + 16*rt + 4*kq + 0..3
  if (WP > 1 && kq >= 4 / WP) return;
  if (EPI != 1) {
#pragma unroll
    for (int rt = 0; rt < R; ++rt)
#pragma unroll
      for (int cb = 0; cb < MB; ++cb)
        store_sums<EPI, true, TO>(c, acc[rt][cb], before[rt][cb], gain[rt], 16 * cb + r, n0 + part0 + 16 * rt + 4 * kq, m, n,
                            n0 / 16 + rt, kq, fa);
  } else {
    const int half_n = n / 2;
    const GatePair gp = gate_pair(fa.act);
#pragma unroll
    for (int rt = 0; rt + 1 < R; rt += 2)
#pragma unroll
      for (int cb = 0; cb < MB; ++cb) {
        const int mm = 16 * cb + r;
        const int nn = n0 / 2 + 16 * (rt / 2) + 4 * kq;
        if (mm >= m) continue;
        TO* dst = c + (size_t)mm * half_n + nn;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = gated_value(acc[rt][cb][i], acc[rt + 1][cb][i], gp);
        if (sizeof(TO) == 2 && fa.wide) {                  // (n is a multiple of 32)
          if (nn < half_n) *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
          continue;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (nn + i < half_n) Num<TO>::store(dst + i, v[i]);
      }
  }
}

static int skinny_rows(int n, int k, bool pairs);

static int g_tune_parts = 0;
extern "C" void rb_tune_parts(int parts) { g_tune_parts = parts; }      // experiments and tests only: 1 or 2 workgroups for a tile of 16 rows; 0 = the built-in choice
static int g_tune_r = 0, g_tune_waves = 0;
extern "C" void rb_tune(int r, int waves) {       // experiments only; 0 = the built-in choice
  g_tune_r = r;
  g_tune_waves = waves;
}

static FoldArgs fold_args(const GemmTokens& x, const GemmAfter& after, const void* c, int n) {
  const uintptr_t all = reinterpret_cast<uintptr_t>(c) | reinterpret_cast<uintptr_t>(after.gain) | reinterpret_cast<uintptr_t>(after.gained);
  return FoldArgs{x.squares, x.rows, x.eps, after.gain, after.gained, after.squares, n % 4 == 0 && (all & 15) == 0 ? 1 : 0, after.w_frag ? 1 : 0,
                  after.epilogue <= 1 ? after.act : nullptr};
}

// Two workgroups for a tile of 16 rows where that still is at most one a compute unit.  A compute unit has so many requests under way and no more, so a
// product of few rows takes as long as the units that have any of them need for their share, whatever is asked for ahead (two or four stages in
// flight a wave: no change at any of 12 sizes); the two halves of a 1 KB block, loaded with the lanes of the other half for the next
// block of depth, halve that share.  us with whole tiles and with halves, 4 tokens: 2,048 rows at K = 2048 4.17 and 3.89, 4096 5.75 and 5.42, 8192 10.2 and 8.8,
// 11008 14.0 and 11.8; 896 rows at 2048 3.87 and 3.61; 16 tokens, 2,048 at 8192 12.6 and 11.4.  More than one a unit lose (2,304 rows at 2048 4.28 and
// 4.57), and so do quarters, whose 64 bytes are half a line (2,048 rows at 2048 5.25, 896 4.01).
// At K < 1280 a wave has one or two stages, and what the first trip waits for is whole tiles' worth anyway: 2,048 rows, 4 / 8 / 16 tokens, whole tiles and halves: K = 512 2.66 / 2.71 /
// 2.89 and 2.70 / 2.85 / 3.04, 768 2.95 / 3.14 / 3.18 and 2.90 / 3.10 / 3.40, 1024 3.32 / 3.54 / 3.54 and 3.15 / 3.40 / 3.84; added to C 512 2.81 / 3.32 / 3.35 and 3.00 / 3.05 / 3.22, 1024 3.39 / 3.58 / 3.71 and
// 3.38 / 3.53 / 3.98.
static int skinny_parts(int m, int n, int k, int epilogue) {
  if (g_tune_parts) return g_tune_parts;
  if (2 * ((n + 15) / 16) > rb_compute_units()) return 1;
  if (k >= 1280) return 2;
  if (k >= 896) return m <= 8 ? 2 : 1;
  if (epilogue == 2) return m > 4 ? 2 : 1;
  return k >= 768 && m > 1 && m <= 8 ? 2 : 1;
}
extern "C" int rb_tune_few_parts(int m, int n, int k, int epilogue) { return skinny_parts(m, n, k, epilogue); }      // for tests: the choice

// Whether a product of 9 to 16 tokens (fragment-major W, tokens as they are) sets its operands aside, r row tiles a wave, `grid` workgroups: us without and with, 9 / 16
// tokens.
//  - One tile, added to C: 4,096 at 14336 24.9 / 27.8 and 22.4 / 26.1, 6,144 at 4096 12.05 / 13.7 and 11.0 / 13.0, 2,560 at 1280 4.74 / 4.84 and 4.19 / 4.35, 3,072 at 512 3.42 / 3.43 and 3.07 / 3.21;
//    but not where most waves have one stage and few tiles follow (4,096 rows at 1024 3.90 / 4.18 and 4.19 / 4.37, 3,072 at 896 16 tokens 3.69 and 3.87).  With the next norm's rows the same at
//    K < 2048: 2,048 at 512 3.63 / 3.64 and 3.20 / 3.36, 2,560 at 1280 4.73 / 4.92 and 4.38 / 4.68, 4,096 at 1024 4.22 / 4.53 and 4.47 / 4.79; 4,096 at 14336 23.0 / 23.4 and 23.2 / 23.8.  Else two
//    stages of some waves alone: 2,560 at 1280 4.04 / 4.25 and 3.93 / 4.29, 6,144 at 4096 10.7 / 12.7 and 11.2 / 13.4.
//  - Two: 8,192 at 8192 33.4 / 33.4 and 29.9 / 30.3, with the next norm's rows 32.0 / 32.4 and 30.2 / 30.4; the gate from K = 4096 on and at 1152 and 1280 (8,192 at 8192 33.3 / 33.6 and 30.0 / 30.6; 2,560 at
//    1280 4.96 / 5.27 and 4.74 / 5.14; 10,304 at 2048, 9 tokens, 10.24 and 10.69); added to C up to four workgroups a compute unit (22,016 at 4608 37.0 / 40.0 and 36.0 / 38.7; 57,344 at 8192 163 / 159 and 178 / 169).
//  - Four, which take 198 registers then: added to C (15,360 at 5120 30.2 / 31.0 and 29.2 / 30.2), and the gate on up to three quarters of the units (10,240 at 8192 35.3 / 36.7 and 33.6 / 35.8;
//    16,384 47.6 / 48.0 and 48.8 / 48.7).  With the next norm's rows there are not enough registers (16,384 at 8192 47.3 / 47.5 and 56.2 / 57.2).
// Captured steps of 12 sequences, 8 layers of the 8B shape 823 and 829 us, 5 of the 70B shape 1,700 and 1,669.  (Two whole stages in registers, or W a stage ahead of the
// tokens, both spelled out: slower than either.)
constexpr bool may_set_aside(int r, int epilogue) { return r == 1 ? epilogue == 0 || epilogue == 2 || epilogue == 3 : r == 2 || epilogue == 1 || epilogue == 2; }
static bool set_aside(int r, int epilogue, int k, long long grid) {
  const long long cus = rb_compute_units();
  if (!may_set_aside(r, epilogue)) return false;
  if (r == 1) {
    if (epilogue == 0) return k >= 1152 && k < 1536;
    return k <= 768 || (k >= 1152 && (epilogue == 2 || k < 2048)) || (epilogue == 2 && grid > cus);
  }
  if (r == 2) return epilogue == 1 ? k >= 4096 || (k >= 1152 && k < 1536) : epilogue == 2 ? grid <= 4 * cus : true;
  return epilogue == 2 || 4 * grid <= 3 * cus;
}

// Blocks of depth that a load of the tokens brings, where a tile of rows is one workgroup's: as many as there is room for, except
//  - tokens that a norm prepared: their sums of squares are waited for first, and what is saved behind that seldom makes up for two rows' addresses and the
//    rotations.  us with a block a load and packed, 4 tokens: 2,048 rows at K = 2048 4.61 and 4.73, 8,192 at 8192 28.4 and 29.4; of gate and way up
//    8,192 at 8192 28.5 and 29.7, 8,192 at 2048 7.87 and 8.02.  It pays above K = 4096 with more tiles than compute units (5,120 at 5120 1 to 5 %) and up to four a unit (27,648 at 5120, 6 tokens, 48.0 and 49.7), and for
//    the gate from K = 3072 on with few tiles (4,096 at 14336 4 %) or, with 5 to 8 tokens, many (57,344 at 8192 2 %);
//  - rows of 16 KB or a multiple: where workgroups share a compute unit, the few lines of tokens that packed loads ask for lie in too few channels of the
//    caches (12,288 rows at K = 8192 5 to 7 %; at 7168, 9216 and 10240 nothing is lost);
//  - four row tiles a wave on nearly every compute unit (15,360 rows at K = 5120 26.2 and 26.7 us; the gate on 192 units, 12,288 at 7168, gains 3 to 5 %, and on 432, 27,648 at
//    5120, 2 to 6 %);
//  - 5 to 8 tokens at K <= 1024 while the tiles are few (3,072 rows at K = 1024 4 to 5 %; at 1152 and 1280 it gains 2 to 7 %) and, at K < 2048, with the next norm's rows, while they are many (2 to 3 %).
// Added to C alone the packed loads gain otherwise, up to 30 %.
static int packed_blocks(int m, int n, int k, int r, int epilogue, bool scaled) {
  if (m > 8) return 1;
  const long long tiles = (n + 15) / 16, cus = rb_compute_units();
  const bool whole16k = k % 8192 == 0, short_of_eight = m > 4 && k <= 1024;
  bool pays;
  if (scaled && epilogue == 1)
    pays = (k >= 3072 && 4 * tiles <= (whole16k ? 3 : k > 4096 ? 5 : 4) * cus) || (m > 4 && k > 4096 && tiles > 2 * cus);
  else if (scaled)
    pays = k > 4096 && tiles > (whole16k ? 2 : 1) * cus && tiles <= 4 * cus;
  else if (epilogue == 2)
    pays = !(short_of_eight && tiles <= cus);
  else if (r == 4)
    pays = epilogue == 3 ? !(whole16k && tiles <= 4 * cus) : epilogue == 1 && (tiles <= 3 * cus || (!whole16k && tiles > 4 * cus));
  else if (epilogue == 3)
    pays = !(whole16k && r == 1 && tiles > 2 * cus) && !(m > 4 && k < 2048 && tiles > 2 * cus && tiles <= 4 * cus);
  else
    pays = !(whole16k && r == 1 && tiles > 2 * cus) && !(short_of_eight && tiles < 2 * cus);
  return !pays ? 1 : m <= 4 ? 4 : 2;
}

// For tests: the choices for a fragment-major product, tokens as they are or prepared by a norm
extern "C" int rb_tune_few_aside(int n, int k, int epilogue) {
  const int r = skinny_rows(n, k, epilogue == 1);
  return set_aside(r, epilogue, k, (n + 16 * r - 1) / (16 * r));
}
extern "C" int rb_tune_few_blocks(int m, int n, int k, int epilogue, int prepared) {
  return k % 128 != 0 || m > 16 ? 1 : packed_blocks(m, n, k, skinny_rows(n, k, epilogue == 1), epilogue, prepared != 0);
}

template <int MB, int R, bool FAST, int EPI, typename TO, bool SCALED>
static int launch_skinny(const GemmTokens& x, const bf16_t* w, void* c, const GemmAfter& after, int m, int n, int k,
                         int n_waves, int k_per_wave, hipStream_t s) {
  const size_t lds = (size_t)(n_waves - 1) * (R * MB * 4 + (SCALED ? MB : 0)) * 64 * sizeof(float);
  RB_REQUIRE(lds <= 64 * 1024, "rb_gemm_bf16: internal: reduction buffer of %zu bytes", lds);
  const int grid = (n + 16 * R - 1) / (16 * R);
  if constexpr (MB == 1 && R == 1 && FAST && !SCALED && (EPI == 0 || EPI == 2 || EPI == EPI_ACT)) {
    if (after.w_frag && skinny_parts(m, n, k, EPI) == 2) {
      (m <= 4   ? gemm_skinny_kernel<1, 1, true, true, EPI, TO, false, 4, 2>
       : m <= 8 ? gemm_skinny_kernel<1, 1, true, true, EPI, TO, false, 2, 2>
                : gemm_skinny_kernel<1, 1, true, true, EPI, TO, false, 1, 2>)<<<2 * grid, n_waves * 64, lds, s>>>(
          x.x, w, (TO*)c, m, n, k, k_per_wave, fold_args(x, after, c, n));
      return 0;
    }
  }
  if (MB == 1 && after.w_frag) {
    constexpr bool MAY = MB == 1 && FAST, MAY_ASIDE = MAY && !SCALED && may_set_aside(R, EPI);
    const int blocks = MAY ? packed_blocks(m, n, k, R, EPI, SCALED) : 1;
    const bool aside = MAY_ASIDE && set_aside(R, EPI, k, grid);
    (blocks == 4   ? gemm_skinny_kernel<MB, R, FAST, MB == 1, EPI, TO, SCALED, MAY ? 4 : 1>
     : blocks == 2 ? gemm_skinny_kernel<MB, R, FAST, MB == 1, EPI, TO, SCALED, MAY ? 2 : 1>
     : aside       ? gemm_skinny_kernel<MB, R, FAST, MB == 1, EPI, TO, SCALED, 1, 1, MAY_ASIDE>
                   : gemm_skinny_kernel<MB, R, FAST, MB == 1, EPI, TO, SCALED, 1>)
        <<<grid, n_waves * 64, lds, s>>>(x.x, w, (TO*)c, m, n, k, k_per_wave, fold_args(x, after, c, n));
  } else
    gemm_skinny_kernel<MB, R, FAST, false, EPI, TO, SCALED, 1>
        <<<grid, n_waves * 64, lds, s>>>(x.x, w, (TO*)c, m, n, k, k_per_wave, fold_args(x, after, c, n));
  return 0;
}

// How K is dealt to the waves of a workgroup.  Fast path: K = 128 * T, the T stages dealt to
// the waves as evenly as they go.  Otherwise the checked path with up to 8 waves.  Measured on the Llama-3-8B
// products at M = 1..8: one stage in flight per wave (U = 1) is as fast as 2 or 4, and 4
// waves beat 8 at K = 4096, 8 beat 4 at K = 14336.  (With W fragment-major again: launched alone, products
// with K = 8192 and more gain up to 10 % from two or four stages in flight; the decode steps they belong to
// lose 4-6 % at the 8B and 70B shapes and gain 1-2 % at hidden sizes of 2,048 and 3,072.  One stage it stays.)
static int skinny_waves(int n, int k, int r, int max_waves) {
  const long long wgs = (n + 16 * r - 1) / (16 * r);
  // 8 waves where K is long, or where every compute unit gets one workgroup at most and so needs
  // more loads in flight of its own (4,096 rows at K = 4096: 8.1-8.3 us against 8.6-9.0 with 4);
  // 4 where several workgroups share a compute unit (6,144 rows: 10.7 against 11.6 with 8)
  int nw = g_tune_waves ? g_tune_waves : ((k >= 8192 || wgs <= rb_compute_units() || max_waves < 4) ? max_waves : 4);
  if (nw > max_waves) nw = max_waves;
  return nw > k / 128 ? k / 128 : nw;
}
template <int MB, int R, int EPI, typename TO, bool SCALED>
static int launch_skinny_u(const GemmTokens& x, const bf16_t* w, void* c, const GemmAfter& after, int m, int n, int k,
                           hipStream_t s) {
  constexpr int max_waves = (R * MB <= 4) ? 8 : (R * MB <= 8 ? 4 : 3);      // bounds the reduction buffer
  if (k % 128 == 0) {
    const int nw = skinny_waves(n, k, R, max_waves);
    return launch_skinny<MB, R, true, EPI, TO, SCALED>(x, w, c, after, m, n, k, nw, 0, s);
  }
  int n_waves = k / 256;
  if (n_waves < 1) n_waves = 1;
  if (n_waves > max_waves) n_waves = max_waves;
  int k_per_wave = (k + n_waves - 1) / n_waves;
  k_per_wave = (k_per_wave + 127) / 128 * 128;
  return launch_skinny<MB, R, false, EPI, TO, SCALED>(x, w, c, after, m, n, k, n_waves, k_per_wave, s);
}

// Row tiles of W per wave (16 R rows per workgroup).  Up to K = 4096 (workgroups of 4 waves, several
// of which share a compute unit) one tile per wave is the fastest at every N from 1024 to 16384
// (measured with 8 tokens, W fragment-major; N = 6144: 11.1 us against 13.5 with two).  From
// K = 8192 on (8 waves) more tiles reuse the token operand better and fewer deal the rows to the 256
// compute units more evenly: the time goes with the rows that the busiest compute unit gets, at
// a price per row that falls with R (about 15 % / R).  57344 rows at K = 8192: R = 4 gives 896
// workgroups, 4 on some compute units and 3 on others, 194 us; R = 2 gives every one 7: 175 us.
// 10240 rows at K = 8192 with one token: R = 1 35 us, R = 2 42; R = 4 takes 31 us by itself (160
// workgroups), but the decode step of that shape is no faster with it (+0.3 % at batch 1, +0.5 % at
// 8, -1.1 % at 16, each the mean of four runs in alternating order), so it is not taken.
// Between K = 4096 and 8192 the same estimate holds: 15,360 rows at K = 5120 with 16 tokens 26.6 us
// with R = 4 against 33.6 with R = 1 (8 tokens: 26.4 against 27.5, one token 26.9 against 26.5),
// 5,120 rows 13.6 with R = 2 against 16.8 (8 tokens: 12.1 against 13.4).
static int skinny_rows(int n, int k, bool pairs) {
  int r = 1;
  if (k > 4096) {
    double best = 0.0;
    const long long cus = rb_compute_units();
    for (int cand = (pairs ? 2 : 1); cand <= 4; cand *= 2) {
      const long long wgs = (n + 16 * cand - 1) / (16 * cand);
      const double cost = (double)((wgs + cus - 1) / cus * 16 * cand) * (1.0 + 0.15 / cand);
      if (best == 0.0 || cost <= best) {
        best = cost;
        r = cand;
      }
    }
  }
  if (g_tune_r) r = g_tune_r;
  return pairs && r < 2 ? 2 : r;
}

int gemm_skinny_waves(int n, int k) { return skinny_waves(n, k, 1, 8); }
bool gemm_skinny_waves_alone(int n, int k) { return skinny_waves(n, k, skinny_rows(n, k, false), 8) == skinny_waves(n, k, 1, 8); }

template <int EPI, typename TO, bool SCALED>
static int dispatch_skinny(const GemmTokens& x, const bf16_t* w, void* c, const GemmAfter& after, int m, int n, int k,
                           hipStream_t s) {
  constexpr bool FOLDS = SCALED || EPI == 2 || EPI == 3;      // compiled for up to 16 tokens only
  const int mb = (m + 15) / 16;
  RB_REQUIRE(!FOLDS || mb == 1, "rb_gemm_bf16: a product that folds its neighbours in takes at most 16 tokens, not %d",
             m);
  const int r = skinny_rows(n, k, EPI == 1);
#define RB_SK(MBV, RV) return launch_skinny_u<MBV, RV, EPI, TO, SCALED>(x, w, c, after, m, n, k, s)
  if (mb == 1) {
    if (r == 4) RB_SK(1, 4);
    if (r == 2) RB_SK(1, 2);
    if (EPI != 1) RB_SK(1, 1);
  }
  if constexpr (!FOLDS) {
    if (mb == 2) {
      if (r == 4) RB_SK(2, 4);
      if (r == 2) RB_SK(2, 2);
      if (EPI != 1) RB_SK(2, 1);
    } else if (mb == 3) {
      if (r == 4) RB_SK(3, 4);
      if (r == 2) RB_SK(3, 2);
      if (EPI != 1) RB_SK(3, 1);
    } else {
      if (r == 4) RB_SK(4, 4);
      if (r == 2) RB_SK(4, 2);
      if (EPI != 1) RB_SK(4, 1);
    }
  }
#undef RB_SK
  RB_REQUIRE(false, "rb_gemm_bf16: internal: no skinny kernel for M=%d R=%d", m, r);
}

// =============================================================================== skinny, tokens resident
// The same product for M <= 64 with the token operand held in registers: a wave owns a
// fixed slice of K (32 * XQ values), loads the tokens' fragments for it once, and then
// streams the W rows of one 16-row tile after the other through the matrix cores, the
// next tile's loads in flight while the current one is multiplied.  Inside the loop W is
// the only thing read from memory.  A workgroup's waves cover adjacent K slices and add
// their sums through LDS.  SCALED and epilogues 2 and 3 as in the kernel above (one workgroup
// covers all of K).
template <int MB, int XQ, int EPI, typename TO, bool SCALED>
__global__ __launch_bounds__(512) void gemm_resident_kernel(const bf16_t* __restrict__ x,
                                                             const bf16_t* __restrict__ w, TO* __restrict__ c,
                                                             int m, int n, int k, int tiles_per_wg, FoldArgs fa) {
  extern __shared__ float red[];      // [2][waves - 1][MB * 4][64], then SCALED: [waves][MB * 16]
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int n_waves = blockDim.x >> 6;
  const int r = lane & 15;
  const int kq = lane >> 4;
  const int n_tiles = (n + 15) / 16;
  const int tile0 = blockIdx.x * tiles_per_wg;
  int t_count = n_tiles - tile0;
  if (t_count > tiles_per_wg) t_count = tiles_per_wg;
  const int k0 = (blockIdx.y * n_waves + wave) * (32 * XQ) + 8 * kq;
  TO* cpart = c + (size_t)blockIdx.y * m * (EPI == 1 ? n / 2 : n);

  if (t_count <= 0) return;
  Frag8 a0[XQ], a1[XQ];
  auto load_tile = [&](Frag8* a, int t) {
    if (fa.w_frag) {
      // fragment-major: the wave's XQ blocks of a tile are XQ KB in a row; read once, past the caches
      int tile = tile0 + t;
      if (tile * 16 >= n) tile = 0;              // results of such rows are never stored
      const bf16_t* p = w + ((size_t)tile * k + (size_t)(blockIdx.y * n_waves + wave) * (32 * XQ)) * 16 + 8 * lane;
#pragma unroll
      for (int j = 0; j < XQ; ++j) a[j].u = load16_stream(p + (size_t)j * 512);
      return;
    }
    int row = (tile0 + t) * 16 + r;
    if (row >= n) row = 0;                       // results of such rows are never stored
    const bf16_t* wrow = w + (size_t)row * k + k0;
#pragma unroll
    for (int j = 0; j < XQ; ++j) a[j].u = load16(wrow + 32 * j);
  };
  load_tile(a0, 0);            // the first rows of W are on their way while the tokens are fetched

  // ---- the tokens' fragments for this wave's slice of K
  Frag8 b[XQ][MB];
  float scale[MB];
#pragma unroll
  for (int cb = 0; cb < MB; ++cb) {
    const int row = 16 * cb + r;
    size_t src = row < m ? row : 0;
    if (fa.rows) src = (size_t)fa.rows[src];
    const bf16_t* xrow = x + src * k + k0;
#pragma unroll
    for (int j = 0; j < XQ; ++j) b[j][cb].u = load16(xrow + 32 * j);
    scale[cb] = 0.f;
    if (SCALED) {
      const int n_sq = (k + 15) / 16;
      scale[cb] = squares_sum(squares_ask(fa.squares_in + src * n_sq, n_sq, wave * 4 + kq, n_waves * 4));
    }
  }
  // SCALED: the waves' shares of the squares meet in LDS behind the first tile's barrier
  float* squares = red + (size_t)2 * (n_waves - 1) * MB * 4 * 64;      // [waves][MB * 16]
  bool scale_known = !SCALED;
  if (SCALED) {
#pragma unroll
    for (int cb = 0; cb < MB; ++cb) {
      scale[cb] += __shfl_xor(scale[cb], 16, RB_WAVE);
      scale[cb] += __shfl_xor(scale[cb], 32, RB_WAVE);
      if (n_waves > 1) {
        if (kq == 0) squares[wave * (MB * 16) + cb * 16 + r] = scale[cb];
      } else {
        scale[cb] = 1.0f / sqrtf(scale[cb] / (float)k + fa.eps);
      }
    }
    if (n_waves == 1) scale_known = true;
  }

  f32x4_t gate[MB];                              // EPI 1: the gate tile's sums wait for the up tile
  auto finish_tile = [&](const Frag8* a, int t) {
    f32x4_t acc[MB];
#pragma unroll
    for (int cb = 0; cb < MB; ++cb) acc[cb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < XQ; ++j)
#pragma unroll
      for (int cb = 0; cb < MB; ++cb) acc[cb] = mfma16(a[j], b[j][cb], acc[cb]);
    // the wave that gathers this tile's sums: tiles of a gate/up pair go to the same one
    const int owner = (EPI == 1 ? (t >> 1) : t) % n_waves;
    if (n_waves > 1) {
      float* buf = red + (size_t)(t & 1) * (n_waves - 1) * MB * 4 * 64;
      if (wave != owner) {
        const int slot = wave < owner ? wave : wave - 1;
        float* dst = buf + (size_t)slot * MB * 4 * 64 + lane;
#pragma unroll
        for (int cb = 0; cb < MB; ++cb)
#pragma unroll
          for (int i = 0; i < 4; ++i) dst[(cb * 4 + i) * 64] = acc[cb][i];
      }
      __syncthreads();
      if (SCALED && !scale_known) {
#pragma unroll
        for (int cb = 0; cb < MB; ++cb) {
          float ss = 0.f;
          for (int ww = 0; ww < n_waves; ++ww) ss += squares[ww * (MB * 16) + cb * 16 + r];
          scale[cb] = 1.0f / sqrtf(ss / (float)k + fa.eps);
        }
        scale_known = true;
      }
      if (wave == owner) {
        for (int ww = 0; ww < n_waves - 1; ++ww) {
          const float* src = buf + (size_t)ww * MB * 4 * 64 + lane;
#pragma unroll
          for (int cb = 0; cb < MB; ++cb)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[cb][i] += src[(cb * 4 + i) * 64];
        }
      }
    }
    if (wave != owner) return;
    if (SCALED) {
#pragma unroll
      for (int cb = 0; cb < MB; ++cb)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[cb][i] *= scale[cb];
    }
    const int tile = tile0 + t;
    if (EPI != 1) {
#pragma unroll
      for (int cb = 0; cb < MB; ++cb) {
        const int mm = 16 * cb + r;
        const int nn = tile * 16 + 4 * kq;
        f32x4_t before = (f32x4_t){0.f, 0.f, 0.f, 0.f}, gain = before;
        if (EPI == 2 || EPI == 3) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if (mm < m && nn + i < n) before[i] = Num<TO>::load(cpart + (size_t)mm * n + nn + i);
            if (EPI == 3 && nn + i < n) gain[i] = fa.gain[nn + i];
          }
        }
        store_sums<EPI, EPI == 2 || EPI == 3, TO>(cpart, acc[cb], before, gain, mm, nn, m, n, tile, kq, fa);
      }
    } else if ((t & 1) == 0) {
#pragma unroll
      for (int cb = 0; cb < MB; ++cb) gate[cb] = acc[cb];
    } else {
      const int half_n = n / 2;
      const GatePair gp = gate_pair(fa.act);
#pragma unroll
      for (int cb = 0; cb < MB; ++cb) {
        const int mm = 16 * cb + r;
        const int nn = (tile >> 1) * 16 + 4 * kq;
        if (mm >= m) continue;
        TO* dst = cpart + (size_t)mm * half_n + nn;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (nn + i < half_n) Num<TO>::store(dst + i, gated_value(gate[cb][i], acc[cb][i], gp));
      }
    }
  };

  int t = 0;
  for (; t + 2 < t_count; t += 2) {              // tiles t + 1 and t + 2 exist: loads are unconditional
    load_tile(a1, t + 1);
    finish_tile(a0, t);
    load_tile(a0, t + 2);
    finish_tile(a1, t + 1);
  }
  if (t + 1 < t_count) {
    load_tile(a1, t + 1);
    finish_tile(a0, t);
    finish_tile(a1, t + 1);
  } else {
    finish_tile(a0, t);
  }
}

static int g_res_tiles = 0, g_res_forced = 0;
extern "C" void rb_tune_resident(int tiles) { g_res_tiles = tiles; }      // experiments only; 0 = built-in
void gemm_resident_forced(int on) { g_res_forced = on; }                  // set by rb_tune_use_resident(2)

template <int MB, int XQ, int EPI, typename TO, bool SCALED>
static int launch_resident(const GemmTokens& x, const bf16_t* w, void* c, const GemmAfter& after, int m, int n, int k,
                           int parts, hipStream_t s) {
  const int slices = k / (32 * XQ);
  const int n_waves = slices / parts;
  const int n_tiles = (n + 15) / 16;
  // tiles per workgroup: as many as give every compute unit one workgroup at most, but no more
  // than 16 (measured: 22016 rows in 230 workgroups of 6 tiles take 35 us, in 344 of 4, which
  // come in two rounds, 44 us; 12288 rows 20 us in 256 workgroups, 31 us in 384; the 128256
  // rows of an output layer are as fast in 501 workgroups of 16 tiles as in 251 of 32)
  const int cus = rb_compute_units();
  int tiles = g_res_tiles ? g_res_tiles : (n_tiles + cus - 1) / cus;
  if (!g_res_tiles && tiles > 16) tiles = 16;
  if (EPI == 1 && (tiles & 1)) tiles += 1;
  const size_t lds = ((size_t)2 * (n_waves - 1) * MB * 4 * 64 + (SCALED ? n_waves * MB * 16 : 0)) * sizeof(float);
  dim3 grid((n_tiles + tiles - 1) / tiles, parts);
  gemm_resident_kernel<MB, XQ, EPI, TO, SCALED>
      <<<grid, n_waves * 64, lds, s>>>(x.x, w, (TO*)c, m, n, k, tiles, fold_args(x, after, c, n));
  return 0;
}

static int resident_depth(int m) { return m <= 16 ? 16 : (m <= 32 ? 8 : 4); }      // XQ

bool gemm_resident_takes(int m, int k, int parts) {
  const int each = 32 * resident_depth(m);
  if (k % each != 0 || parts < 1 || k / each % parts != 0) return false;
  const int n_waves = k / each / parts;
  // With fewer than 7 waves a workgroup has too few loads in flight for the one compute unit it has to
  // itself, and the skinny kernel, several workgroups to a compute unit, is faster (32,768 gated rows at
  // K = 2048: 12.4 us against 13.8 with 4 waves; at K = 3072: 17.3 against 18.4 with 6); forced on
  // (rb_tune_use_resident(2)) it still takes them.
  return n_waves <= 8 && (n_waves >= 7 || g_res_forced != 0);
}

// true if the resident kernel takes these sizes
template <int EPI, typename TO, bool SCALED>
static bool try_resident(const GemmTokens& x, const bf16_t* w, void* c, const GemmAfter& after, int m, int n, int k,
                         int parts, hipStream_t s, int* rc) {
  constexpr bool FOLDS = SCALED || EPI == 2 || EPI == 3;      // compiled for up to 16 tokens and all of K in one workgroup
  const int mb = (m + 15) / 16;
  if (!gemm_resident_takes(m, k, parts)) return false;
  if (EPI == 1 && (n % 32 != 0)) return false;
  if (FOLDS && (mb != 1 || parts != 1)) return false;
  if (mb == 1) {
    *rc = launch_resident<1, 16, EPI, TO, SCALED>(x, w, c, after, m, n, k, parts, s);
    return true;
  }
  if constexpr (!FOLDS) {
    if (mb == 2) *rc = launch_resident<2, 8, EPI, TO, false>(x, w, c, after, m, n, k, parts, s);
    else if (mb == 3) *rc = launch_resident<3, 4, EPI, TO, false>(x, w, c, after, m, n, k, parts, s);
    else *rc = launch_resident<4, 4, EPI, TO, false>(x, w, c, after, m, n, k, parts, s);
    return true;
  }
  return false;
}


// One instance per (epilogue, output type, kind of tokens).  Epilogues 2 and 3 are float32 and
// take plain tokens; prepared tokens go with epilogues 0 and 1.
#define RB_PLAIN(FN, ...)                                                                                  \
  (after.epilogue == 0 && after.act ? (dtype_out == RB_F32 ? FN<EPI_ACT, float, false>(__VA_ARGS__) : FN<EPI_ACT, bf16_t, false>(__VA_ARGS__)) : \
   after.epilogue == 3 ? FN<3, float, false>(__VA_ARGS__)                                                  \
   : after.epilogue == 2 ? FN<2, float, false>(__VA_ARGS__)                                                \
   : after.epilogue == 0 ? (dtype_out == RB_F32 ? FN<0, float, false>(__VA_ARGS__) : FN<0, bf16_t, false>(__VA_ARGS__)) \
                         : (dtype_out == RB_F32 ? FN<1, float, false>(__VA_ARGS__) : FN<1, bf16_t, false>(__VA_ARGS__)))
#define RB_SCALED(FN, ...)                                                                                 \
  (after.epilogue == 0 ? (dtype_out == RB_F32 ? FN<0, float, true>(__VA_ARGS__) : FN<0, bf16_t, true>(__VA_ARGS__)) \
                       : (dtype_out == RB_F32 ? FN<1, float, true>(__VA_ARGS__) : FN<1, bf16_t, true>(__VA_ARGS__)))

int gemm_skinny_launch(const GemmTokens& x, const bf16_t* w, void* c, int dtype_out, const GemmAfter& after, int m,
                       int n, int k, hipStream_t s) {
  if (x.squares) {
    RB_REQUIRE(after.epilogue <= 1, "rb_gemm_bf16: prepared rows go with epilogues 0 and 1, not %d", after.epilogue);
    return RB_SCALED(dispatch_skinny, x, w, c, after, m, n, k, s);
  }
  return RB_PLAIN(dispatch_skinny, x, w, c, after, m, n, k, s);
}

bool gemm_resident_try(const GemmTokens& x, const bf16_t* w, void* c, int dtype_out, const GemmAfter& after, int m,
                       int n, int k, hipStream_t s, int* rc) {
  if (x.squares) {
    if (after.epilogue > 1) return false;
    return RB_SCALED(try_resident, x, w, c, after, m, n, k, 1, s, rc);
  }
  return RB_PLAIN(try_resident, x, w, c, after, m, n, k, 1, s, rc);
}
