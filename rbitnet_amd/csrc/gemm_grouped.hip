// Products in groups: the experts of a routed feed-forward for steps of many tokens.  The step's (token, expert) pairs
// are sorted by expert in runs padded to the tiles' rows (rb_route_choose_units), so that a tile of rows belongs to one expert, and
// the tiles are those of the dense product with direct loads into LDS: the way up reads its rows where the tokens lie (a row of a
// tile is any row of h) and leaves the units of the sorted rows; the way down writes every row to its pair's place.  Gated experts
// keep their gate and up rows interleaved in blocks of 16, as the dense gated product does, and run its epilogue.  Where the
// router's weights multiply the experts' inputs, the sums of the way up are multiplied by them instead, before the units' activation, so that
// the tiles still read the tokens' rows as they are (the whole feed-forward below, gathered first and in routed.hip: 731 us; on the tiles 422).
// Bound by the matrix cores; measured beside the kernels of routed.hip (a wave's operands straight from memory, 64 rows by 64
// channels), 3,782 tokens by 4 of 16 experts, width 2,048, 2,048 units an expert: up and down 728 -> 596 us on the tiles of gemm_dma.h and
// 397 on those of gemm_pingpong.h (runs padded to 256 rows).
#include "api.h"
#include "gemm_dma.h"
#include "gemm_pingpong.h"

template <int BN, int BM, int WN, int WM, int S, int GR, typename TO, int EPI = 0>
static int launch_grouped(const bf16_t* x, const bf16_t* w, TO* c, int m_tiles, int n, int k, const float* act, const GemmGroups& groups,
                          hipStream_t s) {
  constexpr int BK = 64;
  const int n_tiles = (n + BN - 1) / BN;
  const long long tiles = (long long)m_tiles * n_tiles;
  RB_REQUIRE(tiles < (1LL << 30), "rb_routed_experts_tiled: too many tiles");
  const size_t lds = (size_t)S * (BN + BM) * BK * sizeof(bf16_t);
  auto kern = gemm_dma_kernel<BN, BM, WN, WM, BK, S, EPI, TO, true, GR>;
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    RB_REQUIRE(e == hipSuccess, "rb_routed_experts_tiled: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    configured = true;
  }
  kern<<<dim3((unsigned)((tiles + 7) / 8 * 8)), 64 * (BN / WN) * (BM / WM), lds, s>>>(x, w, c, nullptr, m_tiles * BM, n, k, m_tiles, n_tiles,
                                                                                      k / BK, 0, act, groups);
  return 0;
}

// the same on the kernel whose waves take turns; the units' activation is compiled in
template <int BN, int BM, int GR, typename TO, int EPI, bool ACT>
static int launch_grouped_pingpong(const bf16_t* x, const bf16_t* w, TO* c, int m_tiles, int n, int k, const float* act, const GemmGroups& groups,
                                   hipStream_t s) {
  const int n_tiles = (n + BN - 1) / BN;
  const long long tiles = (long long)m_tiles * n_tiles;
  RB_REQUIRE(tiles < (1LL << 30), "rb_routed_experts_tiled: too many tiles");
  const size_t lds = (size_t)2 * (BN + BM) * 64 * sizeof(bf16_t);
  auto kern = gemm_pingpong_kernel<BN, BM, EPI, TO, true, GR, false, ACT>;
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    RB_REQUIRE(e == hipSuccess, "rb_routed_experts_tiled: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    configured = true;
  }
  kern<<<dim3((unsigned)((tiles + 7) / 8 * 8)), 512, lds, s>>>(x, w, c, nullptr, m_tiles * BM, n, k, m_tiles, n_tiles, k / 64, 0, act, groups);
  return 0;
}

extern "C" int rb_routed_experts_tiled(const void* h, int n_tokens, int top, const int32_t* row_pair, const int32_t* tile_expert, int unit,
                                       int max_rows, int gated, const void* w_up, const void* w_down, const float* act, void* y, float* out,
                                       int n_experts, int width, int ff, const float* weight, void* stream) {
  RB_RECORDED(rb_routed_experts_tiled(h, n_tokens, top, row_pair, tile_expert, unit, max_rows, gated, w_up, w_down, act, y, out, n_experts,
                                      width, ff, weight, stream));
  RB_REQUIRE(n_tokens >= 0 && top > 0 && n_experts > 0 && width > 0 && ff > 0 && width % 64 == 0 && ff % 64 == 0,
             "rb_routed_experts_tiled: bad sizes T=%d top=%d experts=%d width=%d ff=%d (sizes are multiples of 64)", n_tokens, top, n_experts,
             width, ff);
  RB_REQUIRE((unit == 64 || unit == 128 || unit == 256) && max_rows >= 0 && max_rows % unit == 0,
             "rb_routed_experts_tiled: runs padded to %d rows not supported (64, 128, 256)", unit);
  // byte offsets inside a tile's operands are 32-bit; those of the gathered rows count from h's first
  RB_REQUIRE((long long)n_tokens * width * 2 < (1LL << 32) && 256LL * width * 2 < (1LL << 32) && 256LL * ff * 2 < (1LL << 32),
             "rb_routed_experts_tiled: %d tokens of %d numbers are too many", n_tokens, width);
  RB_REQUIRE(act != nullptr || gated, "rb_routed_experts_tiled: the units need their activation's numbers");
  auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  RB_REQUIRE(aligned(h) && aligned(w_up) && aligned(w_down) && aligned(y) && aligned(out), "rb_routed_experts_tiled: operands must be 16-byte aligned");
  if (n_tokens == 0 || max_rows == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const GemmGroups groups = {tile_expert, row_pair, top, weight};
  const int m_tiles = max_rows / unit;
  const bf16_t *x = (const bf16_t*)h, *wu = (const bf16_t*)w_up, *wd = (const bf16_t*)w_down;
  bf16_t* yb = (bf16_t*)y;
  int rc;
#define GR_PINGPONG(BN, BM)                                                                                                      \
  do {                                                                                                                           \
    if (gated) rc = launch_grouped_pingpong<BN, BM, 1, bf16_t, 1, false>(x, wu, yb, m_tiles, 2 * ff, width, act, groups, s);     \
    else rc = launch_grouped_pingpong<BN, BM, 1, bf16_t, 0, true>(x, wu, yb, m_tiles, ff, width, act, groups, s);                \
    if (!rc) rc = launch_grouped_pingpong<BN, BM, 2, float, 0, false>(yb, wd, out, m_tiles, width, ff, nullptr, groups, s);      \
  } while (0)
  if (unit == 256) {
    GR_PINGPONG(256, 256);
  } else if (unit == 128) {
    GR_PINGPONG(256, 128);
  } else {
    if (gated) rc = launch_grouped<128, 64, 32, 64, 3, 1, bf16_t, 1>(x, wu, yb, m_tiles, 2 * ff, width, act, groups, s);
    else rc = launch_grouped<128, 64, 32, 64, 3, 1, bf16_t>(x, wu, yb, m_tiles, ff, width, act, groups, s);
    if (!rc) rc = launch_grouped<128, 64, 32, 64, 3, 2, float>(yb, wd, out, m_tiles, width, ff, nullptr, groups, s);
  }
#undef GR_PINGPONG
  if (rc) return rc;
  RB_LAUNCH_CHECK();
  return 0;
}
