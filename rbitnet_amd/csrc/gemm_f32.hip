// Float32 products of many tokens on the float32 MFMA (float32 inputs, products and sums; no reduced-precision mode) with tiles that
// go from memory straight into LDS: instances of the kernel in gemm_dma.h.  Bound by the matrix cores: v_mfma_f32_32x32x2_f32 takes
// 16 times as long as bfloat16 for the same product, 157 TFLOP/s at the most, so loads and LDS (a 16-byte read serves four
// MFMAs) are easily covered and what counts is how evenly the outputs are dealt to the compute units.  Measured beside the kernel
// that stages 128 x 128 tiles through registers and stores them depth-major (gemm_generic.hip, still there for K % 32 != 0), W
// fragment-major, 1,286 tokens: 3,072 rows at K = 8192 1,128 -> 525 us (57 -> 123 TFLOP/s), at K = 3072 428 -> 198,
// 5,120 rows 454 -> 353, 16,384 rows 1,241 -> 1,032, 128,256 rows 9.6 -> 7.8 ms; 131 tokens by 5,120 rows 249 -> 63.
#include "api.h"
#include "tune.h"
#include "gemm_dma.h"

static int g_f32_tile = 0;
// experiments only: 0 = the built-in choice, 1..4 = a tile of the list below, -1 = the kernel staged through registers
extern "C" void rb_tune_f32_tile(int tile) { g_f32_tile = tile; }

template <int BN, int BM, int WN, int WM, int S, bool WF>
static int launch_f32_dma(const float* x, const float* w, float* c, int m, int n, int k, hipStream_t s) {
  constexpr int BK = 64;                                   // 32 floats
  const int m_tiles = (m + BM - 1) / BM, n_tiles = (n + BN - 1) / BN;
  const long long tiles = (long long)m_tiles * n_tiles;
  RB_REQUIRE(tiles < (1LL << 30), "rb_gemm_generic: too many tiles");
  const size_t lds = (size_t)S * (BN + BM) * BK * sizeof(bf16_t);
  auto kern = gemm_dma_kernel<BN, BM, WN, WM, BK, S, 0, float, WF, 0, true>;
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    RB_REQUIRE(e == hipSuccess, "rb_gemm_generic: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    configured = true;
  }
  kern<<<dim3((unsigned)((tiles + 7) / 8 * 8)), 64 * (BN / WN) * (BM / WM), lds, s>>>(
      reinterpret_cast<const bf16_t*>(x), reinterpret_cast<const bf16_t*>(w), c, nullptr, m, n, 2 * k, m_tiles, n_tiles, 2 * k / BK,
      nullptr, GemmGroups{nullptr, nullptr, 1});
  return 0;
}

// The time goes with the outputs that the busiest compute unit computes, at a price per output that is a little higher for smaller
// tiles (2,048 tokens by 16,384 rows at K = 3072, which every tile divides: 1,444, 1,507, 1,572 and 1,437 us in this order).
struct F32Tile {
  int bn, bm;
  double per_output;
};
static const F32Tile F32_TILES[] = {{128, 128, 1.0}, {128, 64, 1.04}, {64, 64, 1.09}, {256, 128, 0.995}};

static int pick_f32_tile(int m, int n) {
  int best = 0;
  double least = 0.0;
  const long long cus = rb_compute_units();
  for (int i = 0; i < 4; ++i) {
    const F32Tile& t = F32_TILES[i];
    const long long tiles = (long long)((m + t.bm - 1) / t.bm) * ((n + t.bn - 1) / t.bn);
    const double cost = (double)((tiles + cus - 1) / cus) * t.bn * t.bm * t.per_output;
    if (i == 0 || cost < least) {
      least = cost;
      best = i;
    }
  }
  return best;
}

bool gemm_f32_dma_try(const float* x, const float* w, bool w_frag, float* c, int m, int n, int k, hipStream_t s, int* rc) {
  if (g_f32_tile < 0 || k % 32 != 0 || (w_frag && n % 16 != 0)) return false;
  // 16 bytes a lane and load, and byte offsets inside a tile of 32 bits
  if (((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) != 0 || 256LL * k * 4 >= (1LL << 32)) return false;
  const int tile = g_f32_tile > 0 ? g_f32_tile - 1 : pick_f32_tile(m, n);
#define F32_GO(BN, BM, WN, WM, S)                                               \
  *rc = w_frag ? launch_f32_dma<BN, BM, WN, WM, S, true>(x, w, c, m, n, k, s)   \
               : launch_f32_dma<BN, BM, WN, WM, S, false>(x, w, c, m, n, k, s)
  switch (tile) {
    case 0: F32_GO(128, 128, 64, 64, 2); break;
    case 1: F32_GO(128, 64, 64, 32, 3); break;
    case 2: F32_GO(64, 64, 32, 32, 4); break;
    default: F32_GO(256, 128, 64, 64, 2); break;
  }
#undef F32_GO
  return true;
}
