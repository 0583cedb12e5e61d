// Several products of a few tokens in one launch: C_i = X_i W_i^T, bfloat16 operands, each with inputs, a depth, a matrix, outputs
// and an end of its own.  A layer's projections that do not wait for each other (the inputs of time mixing and what its decays are made
// from; a large product and the low-rank one beside it) were launches one after the other, and a product of 16 to 1,024 rows with 4 tokens at
// K = 2048 costs 3.8 to 5 us whatever it reads (4 MB: 0.6 us of memory's time): its boundary, two trips to memory, the waves' sums.
// The same kernel as gemm_skinny_kernel with one row tile a wave: K / 128 stages dealt to the waves in a row, sums through LDS in their order.
// Sums are those of a product alone: each has the waves that it would have by itself.
// Measured in captured steps of 4 tokens: 6,160 and 256 rows 6.8 + 4.3 us in two launches, 6.6 in one; five of 1,024 and 64 rows and the tanh behind the
// last, 19 + 10 us in six launches, 4.2 in one.  In a chain of launches that read W from memory, 4 tokens, K = 2048: 7.2 for 10.4, 6.8 for 20.2.
#include "api.h"
#include "gemm_internal.h"

namespace {

constexpr int MOST = RB_GROUP_PRODUCTS;
enum { END_F32 = 0, END_BF16 = 1, END_TANH = 2 };          // tanh: bfloat16(tanh(sum))
struct Dealt {
  RbGroupProduct p;
  int waves;                                                // of a workgroup, as if the product were alone
  int base, extra;                                          // stages of 128 of every wave; the first `extra` waves have one more
  int first;                                                // row tiles of the products in front of it
};
struct Group {
  int count;
  int end[MOST];                                            // row tiles up to and with this product
  Dealt of[MOST];
};

// XP: see RowPack.  ASIDE (a block a load): what was loaded is moved out of the way before it is multiplied, so that the next stage's W is asked for while the tokens
// of this one are waited for.
template <bool WF, int XP, bool ASIDE = false>
__global__ __launch_bounds__(512) void gemm_group_kernel(const Group g, int m) {
  extern __shared__ __attribute__((aligned(16))) float red[];      // [waves - 1][64] pieces of four sums
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, kq = lane >> 4;
  int i = 0;
  while (i + 1 < g.count && (int)blockIdx.x >= g.end[i]) ++i;
  const Dealt of = g.of[i];
  const RbGroupProduct p = of.p;
  const int k = p.k, n_waves = of.waves;
  const int n0 = 16 * ((int)blockIdx.x - of.first);
  const bf16_t* w = (const bf16_t*)p.w;
  const bf16_t* wrow = WF ? w + (size_t)n0 * k + 8 * lane : w + (size_t)(n0 + r < p.n ? n0 + r : 0) * k + 8 * kq;
  const int row = RowPack<XP>::row(r);
  const bf16_t* xrow = (const bf16_t*)p.x + (size_t)(row < m ? row : 0) * k + RowPack<XP>::depth(r) + 8 * kq;
  const int stages = of.base + (wave < of.extra ? 1 : 0), begin = 128 * (wave * of.base + (wave < of.extra ? wave : of.extra));
  f32x4_t acc = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  Frag8 a[4], b[4 / XP];
  auto load_stage = [&](int st) {
    const int ks = begin + 128 * st;
#pragma unroll
    for (int j = 0; j < 4; ++j) a[j].u = WF ? load16_stream(wrow + (size_t)(ks + 32 * j) * 16) : load16(wrow + ks + 32 * j);
#pragma unroll
    for (int j = 0; j < 4 / XP; ++j) b[j].u = load16(xrow + ks + 32 * XP * j);
  };
  auto multiply_stage = [&]() {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (XP == 1 && !ASIDE) acc = mfma16(a[j], b[j], acc);
      else acc = mfma16(a[j], RowPack<XP>::block(b, j), acc);
    }
  };
  if (wave < n_waves) {                                     // (the host gives a product no more waves than stages)
    load_stage(0);
    for (int st = 1; st < stages; ++st) {
      multiply_stage();
      load_stage(st);
    }
    multiply_stage();
  }
  if (blockDim.x > 64) {
    if (wave > 0 && wave < n_waves) *reinterpret_cast<f32x4_t*>(red + (wave - 1) * 256 + 4 * lane) = acc;
    __syncthreads();
    if (wave > 0) return;
    for (int v = 0; v < n_waves - 1; ++v) acc += *reinterpret_cast<const f32x4_t*>(red + v * 256 + 4 * lane);
  }
  if (r >= m) return;
  const int nn = n0 + 4 * kq;                               // token r, rows nn .. + 3
  if (p.end == END_TANH) {
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = tanhf(acc[e]);
  }
  if (p.end == END_F32) {
    float* c = (float*)p.c + (size_t)r * p.n + nn;
    if (p.n % 4 == 0) {
      if (nn < p.n) *reinterpret_cast<f32x4_t*>(c) = acc;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (nn + e < p.n) c[e] = acc[e];
    }
  } else {
    bf16_t* c = (bf16_t*)p.c + (size_t)r * p.n + nn;
    if (p.n % 4 == 0) {
      if (nn < p.n) *reinterpret_cast<uint2*>(c) = make_uint2(pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3]));
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (nn + e < p.n) c[e] = f32_to_bf16(acc[e]);
    }
  }
}

}  // namespace

// Whether m tokens of depth k can go in one launch (more tokens have kernels that deal a product's tiles out better).
extern "C" int rb_gemm_bf16_group_ok(int m, int k) { return m >= 1 && m <= 16 && k >= 128 && k % 128 == 0; }

// Whether a product of n rows is as fast among others as alone, and the same bits: where it has one row tile a wave alone as well, or as many
// waves with more of them.  Groups / their products one after another, 1 and 16 tokens: K = 4096, 6,160 and 256 rows 11.6/15.0 and 13.7/20.4 us, 4,096 twice
// 13.5/15.0 and 14.6/16.9, 64 twice 5.5/10.0 and 7.3/13.6; K = 8192, 8,192 and 1,024 rows 30.9/41.0 and 36.6/44.6; K = 256, five of 1,024 and 64 3.4/11.4 and
// 3.6/12.5.  Left out: K = 5120 with 16,384 rows twice (four row tiles a wave alone) 54.5/55.5 and 69.0/56.1, and 3584 or 4096 with more than
// 8,192 rows (resident tokens: other sums) 43.8/47.6 and 52.4/52.3.
extern "C" int rb_gemm_bf16_group_pays(int m, int n, int k) { return rb_gemm_bf16_group_ok(m, k) && n > 0 && gemm_sums_alone_alike(m, n, k); }

// How a launch of `tiles` row tiles, the longest depth k, loads its tokens (fragment-major W): 4 or 2 blocks of depth a load, or one, 1: multiplied where it was loaded,
// or 0: set aside.  The same bits.  us with 1, 0 and packed loads, W from beyond the caches (and as it was: an operand through RowPack's function in any case, every wave
// dividing its product's stages; before that without packed loads):
//  - short depths on few tiles are one trip to memory, and what stands in front of the multiplications is what counts: K = 768, 768 rows twice and 48, 8 tokens 3.07, 3.28, 3.31
//    (3.44; 3.17), 9 tokens 3.12, 3.34 (3.46; 3.22); K = 1024, 1,024 and 32 twice, 12 tokens 3.40, 3.62 (3.80; 3.55); on many tiles K = 256, five of 1,024, 4 tokens 3.17, 2.83, 2.82
//    (2.95; 3.19), 9 tokens 3.22, 2.95 (2.99; 3.32);
//  - K = 2048, five of 1,024 and 64 rows, 8 tokens 7.34, 7.22, 7.72 (7.31; 7.32); K = 2560, 2,560 twice and 48, 4 tokens 8.11, 8.05, 7.91 (7.98; 8.26);
//    K = 4096, 6,160 and 256, 5 tokens 12.02, 12.01, 12.15 (12.35; 12.01), 8 tokens 12.43, 12.05, 12.50 (12.34; 12.50);
//  - rows of 16 KB on shared compute units: K = 8192, 6,144 and 1,024 rows, 8 tokens 23.6, 24.6, 24.2 (24.1; 23.8), 9 tokens 24.1, 25.1 (25.0; 24.3).
static int group_form(int m, int k, long long tiles) {
  const long long cus = rb_compute_units();
  const bool whole16k = k % 8192 == 0;
  if (whole16k && 2 * tiles > 3 * cus) return 1;
  if (m > 8) return tiles >= cus && k < 2048 && (k <= 256 || k >= 1280) ? 0 : 1;
  if (k < 1024 ? tiles <= cus : m > 4 && k < 2048 && 2 * tiles <= cus) return 1;
  if (k >= 2048 && !whole16k && (k < 2560 || (m > 4 && tiles > cus))) return 0;
  return m <= 4 ? 4 : 2;
}
extern "C" int rb_tune_group_form(int m, int k, int tiles) { return group_form(m, k, tiles); }      // for tests: the choice

extern "C" int rb_gemm_bf16_group(const RbGroupProduct* products, int count, int w_layout, int m, void* stream) {
  RB_REQUIRE(products != nullptr && count >= 1 && count <= MOST, "rb_gemm_bf16_group: %d products (1 to %d)", count, MOST);
  RbGroupProduct all[MOST];
  for (int i = 0; i < count; ++i) all[i] = products[i];
  RB_RECORDED(rb_gemm_bf16_group(all, count, w_layout, m, stream));
  Group g;
  g.count = count;
  RB_REQUIRE(w_layout == 0 || w_layout == 1, "rb_gemm_bf16_group: W layout %d", w_layout);
  long long tiles = 0;
  for (int i = 0; i < count; ++i) {
    const RbGroupProduct& p = products[i];
    RB_REQUIRE(m == 0 || rb_gemm_bf16_group_ok(m, p.k), "rb_gemm_bf16_group: M=%d K=%d is not for it", m, p.k);
    RB_REQUIRE(p.x && p.w && p.c && p.n > 0 && p.end >= END_F32 && p.end <= END_TANH && (w_layout == 0 || p.n % 16 == 0),
               "rb_gemm_bf16_group: product %d of %d rows, layout %d, end %d", i, p.n, w_layout, p.end);
    RB_REQUIRE(((reinterpret_cast<uintptr_t>(p.x) | reinterpret_cast<uintptr_t>(p.w) | reinterpret_cast<uintptr_t>(p.c)) & 15) == 0,
               "rb_gemm_bf16_group: product %d is not aligned to 16 bytes", i);
    g.of[i].p = p;
    g.of[i].first = (int)tiles;
    tiles += (p.n + 15) / 16;
    RB_REQUIRE(tiles <= 1 << 24, "rb_gemm_bf16_group: too many rows");
    g.end[i] = (int)tiles;
  }
  if (m == 0) return 0;
  // every product has the waves that it has alone with one row tile a wave; the others of its workgroups wait at the barrier
  int waves = 1;
  for (int i = 0; i < count; ++i) {
    Dealt& of = g.of[i];
    of.waves = gemm_skinny_waves(of.p.n, of.p.k);
    of.base = of.p.k / 128 / of.waves;
    of.extra = of.p.k / 128 % of.waves;
    if (of.waves > waves) waves = of.waves;
  }
  const size_t lds = (size_t)(waves - 1) * 256 * sizeof(float);
  int depth = 0;
  for (int i = 0; i < count; ++i)
    if (g.of[i].p.k > depth) depth = g.of[i].p.k;
  const int form = group_form(m, depth, tiles);
  (!w_layout   ? gemm_group_kernel<false, 1>
   : form == 4 ? gemm_group_kernel<true, 4>
   : form == 2 ? gemm_group_kernel<true, 2>
   : form == 1 ? gemm_group_kernel<true, 1>
               : gemm_group_kernel<true, 1, true>)<<<(int)tiles, waves * 64, lds, (hipStream_t)stream>>>(g, m);
  RB_LAUNCH_CHECK();
  return 0;
}
