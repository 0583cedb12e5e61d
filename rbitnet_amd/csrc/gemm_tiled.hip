// Products with many tokens (prefill) and with 17..64 tokens: tiles of W and of the tokens
// through LDS, MFMA 32x32x16 bf16, float32 accumulation.  The tokens are the row operand of the
// MFMA and W's rows its columns, so that the lanes of a wave hold consecutive outputs of a token.
//
// Epilogue 1 expects W with gate and up rows interleaved in blocks of 16 and writes
// silu(gate) * up (llama/model.rs:297-302 of the reference) instead of the two products.
//
// Reference loop: y[o] = sum_i W[i + o * n_in] * x[i]  (llama/model.rs:67-91).
#include <type_traits>

#include "api.h"
#include "tune.h"
#include "gemm_internal.h"
#include "gemm_dma.h"
#include "gemm_pingpong.h"

// Adds up the [M, N] slabs of partial sums that the K slices of a product wrote, in slice
// order (the same order whatever else runs), and converts to the output type.
template <typename TO>
__global__ void gemm_sum_slabs_kernel(const float* __restrict__ slabs, TO* __restrict__ c, int parts, size_t count,
                                      const float* __restrict__ act) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  float v = 0.f;
  for (int p = 0; p < parts; ++p) v += slabs[(size_t)p * count + i];
  if (act) {                               // an activation belongs to the whole sum: here, not in the slices
    const XieluPair a = xielu_pair(act);
    v = xielu_value(v, a.ap, a.an);
  }
  Num<TO>::store(c + i, v);
}

#define TG_BK 64
#define TG_LD 72          // bf16 elements per LDS row: 64 + 8 of padding, so that the 16 lanes
                          // of a quarter wave read 16 different 16-byte bank groups

template <int BN, int BM, int WN, int WM, int P, int EPI, bool KTAIL, typename TO>
__global__ __launch_bounds__(64 * (BN / WN) * (BM / WM)) void gemm_tiled_kernel(const bf16_t* __restrict__ x,
                                                         const bf16_t* __restrict__ w, TO* __restrict__ c,
                                                         int m, int n, int k, int m_tiles, int n_tiles,
                                                         const float* __restrict__ act) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  constexpr int TN = WN / 32, TM = WM / 32;
  constexpr int WAVES_N = BN / WN;
  constexpr int NT = 64 * (BN / WN) * (BM / WM);      // threads: one wave per WN x WM piece of the tile
  constexpr int W_CHUNKS = BN * 8 / NT, X_CHUNKS = BM * 8 / NT;
  static_assert(BN * 8 % NT == 0 && BM * 8 % NT == 0 && NT % 8 == 0, "tile does not divide among the threads");
  bf16_t* ws = reinterpret_cast<bf16_t*>(smem);                      // [2][BN][TG_LD]
  bf16_t* xs = ws + 2 * BN * TG_LD;                                  // [2][BM][TG_LD]

  int mt, nt;
  if (!tile_of_workgroup(m_tiles, n_tiles, &mt, &nt)) return;
  const int m0 = mt * BM;
  const int n0 = nt * BN;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wn0 = (wave % WAVES_N) * WN;
  const int wm0 = (wave / WAVES_N) * WM;
  const int l32 = lane & 31;
  const int g = lane >> 5;

  f32x16_t acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // ---- pipeline: tile kt is multiplied out of LDS while tiles kt + 1 .. kt + P - 1 are on
  // their way from memory in registers (P - 1 tiles of latency hidden) and one of them is
  // moved into the other LDS buffer.  Loads carry no conditions: rows beyond N or M are read
  // from the last row and never stored, chunks beyond K are read from the last chunk and
  // zeroed on their way into LDS.  (With conditions the compiler cannot count outstanding
  // loads and waits for all of them.)
  uint4 wreg[P][W_CHUNKS], xreg[P][X_CHUNKS];
  // addresses: a 64-bit base per tile (the same for the whole workgroup) plus a 32-bit
  // element offset per chunk; a tile spans at most 256 rows, so the offsets fit
  const bf16_t* wtile = w + (size_t)n0 * k;
  const bf16_t* xtile = x + (size_t)m0 * k;
  uint32_t woff[W_CHUNKS], xoff[X_CHUNKS];
#pragma unroll
  for (int i = 0; i < W_CHUNKS; ++i) {
    int row = (tid + NT * i) / 8;
    if (n0 + row > n - 1) row = n - 1 - n0;
    woff[i] = (uint32_t)row * (uint32_t)k;
  }
#pragma unroll
  for (int i = 0; i < X_CHUNKS; ++i) {
    int row = (tid + NT * i) / 8;
    if (m0 + row > m - 1) row = m - 1 - m0;
    xoff[i] = (uint32_t)row * (uint32_t)k;
  }
  const int kc = (tid % 8) * 8;             // this thread's chunk offset inside a tile (the same for all i)
  auto load_global = [&](int slot, int kt) {
    int col = kt * TG_BK + kc;
    if (col > k - 8) col = k - 8;           // beyond K: any valid address; the data is zeroed in store_lds
#pragma unroll
    for (int i = 0; i < W_CHUNKS; ++i) wreg[slot][i] = load16(wtile + (woff[i] + (uint32_t)col));
#pragma unroll
    for (int i = 0; i < X_CHUNKS; ++i) xreg[slot][i] = load16(xtile + (xoff[i] + (uint32_t)col));
  };
  auto store_lds = [&](int slot, int kt) {
    const int buf = kt & 1;
    const bool in = !KTAIL || kt * TG_BK + kc < k;
#pragma unroll
    for (int i = 0; i < W_CHUNKS; ++i) {
      const int q = tid + NT * i;
      *reinterpret_cast<uint4*>(ws + ((size_t)buf * BN + q / 8) * TG_LD + kc) = in ? wreg[slot][i] : zero16();
    }
#pragma unroll
    for (int i = 0; i < X_CHUNKS; ++i) {
      const int q = tid + NT * i;
      *reinterpret_cast<uint4*>(xs + ((size_t)buf * BM + q / 8) * TG_LD + kc) = in ? xreg[slot][i] : zero16();
    }
  };
  auto multiply = [&](int kt) {
    const bf16_t* wb = ws + (size_t)(kt & 1) * BN * TG_LD;
    const bf16_t* xb = xs + (size_t)(kt & 1) * BM * TG_LD;
    if (NT <= 256) {
      // fragments of k-step ks + 1 are requested from LDS before the MFMAs of k-step ks
      Frag8 a[2][TN], b[2][TM];
      auto load_frags = [&](int buf2, int ks) {
#pragma unroll
        for (int i = 0; i < TN; ++i)
          a[buf2][i].u = *reinterpret_cast<const uint4*>(wb + (size_t)(wn0 + 32 * i + l32) * TG_LD + ks * 16 + g * 8);
#pragma unroll
        for (int j = 0; j < TM; ++j)
          b[buf2][j].u = *reinterpret_cast<const uint4*>(xb + (size_t)(wm0 + 32 * j + l32) * TG_LD + ks * 16 + g * 8);
      };
      load_frags(0, 0);
#pragma unroll
      for (int ks = 0; ks < TG_BK / 16; ++ks) {
        if (ks + 1 < TG_BK / 16) load_frags((ks + 1) & 1, ks + 1);
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
          for (int j = 0; j < TM; ++j) acc[i][j] = mfma32(b[ks & 1][j], a[ks & 1][i], acc[i][j]);
      }
    } else {
      // 8 waves: two per SIMD cover each other's LDS latency, and registers are scarce
#pragma unroll
      for (int ks = 0; ks < TG_BK / 16; ++ks) {
        Frag8 a[TN], b[TM];
#pragma unroll
        for (int i = 0; i < TN; ++i)
          a[i].u = *reinterpret_cast<const uint4*>(wb + (size_t)(wn0 + 32 * i + l32) * TG_LD + ks * 16 + g * 8);
#pragma unroll
        for (int j = 0; j < TM; ++j)
          b[j].u = *reinterpret_cast<const uint4*>(xb + (size_t)(wm0 + 32 * j + l32) * TG_LD + ks * 16 + g * 8);
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
          for (int j = 0; j < TM; ++j) acc[i][j] = mfma32(b[j], a[i], acc[i][j]);
      }
    }
  };

  const int k_tiles = (k + TG_BK - 1) / TG_BK;
  // tiles beyond the last are loaded as well (clamped) and never stored: the loop body stays
  // free of conditions on loads
#pragma unroll
  for (int sl = 0; sl < P; ++sl) load_global(sl, sl);
  store_lds(0, 0);
  __syncthreads();
  int kt = 0;
  for (; kt + P <= k_tiles; kt += P) {        // P iterations per trip, so that the register slots are static
#pragma unroll
    for (int u = 0; u < P; ++u) {
      // slot u held tile kt + u (now in LDS): reuse it for tile kt + u + P
      load_global(u, kt + u + P);
      multiply(kt + u);
      if (kt + u + 1 < k_tiles) store_lds((u + 1) % P, kt + u + 1);
      __syncthreads();
    }
  }
#pragma unroll
  for (int u = 0; u < P; ++u) {               // the last k_tiles % P tiles
    if (kt + u < k_tiles) {
      multiply(kt + u);
      if (kt + u + 1 < k_tiles) store_lds((u + 1) % P, kt + u + 1);
      __syncthreads();
    }
  }

  // ---- lane holds, per (i, j): W row n0 + wn0 + 32 i + l32, tokens base + 8 (e / 4) + 4 g + e % 4
  const bool has_act = EPI == 0 && act != nullptr;
  XieluPair xa = {0.f, 0.f};
  if (has_act) xa = xielu_pair(act);
  const GatePair gp = gate_pair(EPI == 1 ? act : nullptr);
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j)
      store_piece<EPI, TO>(acc[i][j], c, nullptr, n0 + wn0 + 32 * i, l32, m0 + wm0 + 32 * j + 4 * g, m, n, has_act, xa.ap, xa.an, gp);
}

// ---------------------------------------------------------------------------------------
// The rows of W that a launch computes: all of them, or where a product is two launches (see TilePlan) those of one.
struct RowRange {
  int first, last;
};

template <int BN, int BM, int WN, int WM, int BK, int S, int EPI, typename TO, bool WF>
static int launch_dma_cfg(const bf16_t* x, const bf16_t* w, void* c, int m, int n, int k, RowRange rows, hipStream_t s,
                          int parts = 1, float* slabs = nullptr, const float* act = nullptr) {
  const int m_tiles = (m + BM - 1) / BM, n_tiles = (rows.last - rows.first + BN - 1) / BN;
  RB_REQUIRE(parts >= 1 && (k / BK) % parts == 0 && (parts == 1 || (slabs && EPI == 0)),
             "rb_gemm_bf16: internal: bad K split %d", parts);
  const long long tiles = (long long)m_tiles * n_tiles;
  RB_REQUIRE(tiles < (1LL << 30), "rb_gemm_bf16: too many tiles");
  RB_REQUIRE(k % BK == 0, "rb_gemm_bf16: the direct-to-LDS kernel needs K=%d to be a multiple of %d", k, BK);
  // byte offsets inside a tile are 32-bit
  RB_REQUIRE((long long)(BN > BM ? BN : BM) * k * 2 < (1LL << 32), "rb_gemm_bf16: K=%d too long for this kernel", k);
  const size_t lds = (size_t)S * (BN + BM) * BK * sizeof(bf16_t);
  RB_REQUIRE(!WF || (BN % 32 == 0 && n % 16 == 0), "rb_gemm_bf16: fragment-major W needs N=%d to be a multiple of 16", n);
  auto kern = gemm_dma_kernel<BN, BM, WN, WM, BK, S, EPI, TO, WF>;
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    RB_REQUIRE(e == hipSuccess, "rb_gemm_bf16: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    configured = true;
  }
  const dim3 grid((unsigned)((tiles + 7) / 8 * 8), (unsigned)parts);
  RB_REQUIRE(act == nullptr || (EPI <= 1 && c != nullptr), "rb_gemm_bf16: internal: an activation or a gate's numbers go with epilogues 0 and 1 and an output");
  kern<<<grid, 64 * (BN / WN) * (BM / WM), lds, s>>>(x, w, (TO*)c, parts > 1 ? slabs : nullptr, m, n, k, m_tiles,
                                                      n_tiles, k / BK / parts, rows.first, act, GemmGroups{nullptr, nullptr, 1});
  if (parts > 1 && c != nullptr) {      // without c the caller adds the slabs up itself
    const size_t count = (size_t)m * n;
    gemm_sum_slabs_kernel<TO><<<(unsigned)((count + 255) / 256), 256, 0, s>>>(slabs, (TO*)c, parts, count, EPI == 0 ? act : nullptr);
  }
  return 0;
}

// the same on the kernel whose waves take turns; an activation is compiled in
template <int BN, int BM, int EPI, typename TO, bool WF, bool ACT>
static int launch_pingpong_kernel(const bf16_t* x, const bf16_t* w, void* c, int m, int n, int k, RowRange rows, hipStream_t s, int parts,
                                  float* slabs, const float* act) {
  const int m_tiles = (m + BM - 1) / BM, n_tiles = (rows.last - rows.first + BN - 1) / BN;
  RB_REQUIRE(parts >= 1 && k % 64 == 0 && (k / 64) % parts == 0 && (parts == 1 || (slabs && EPI == 0 && !ACT)),
             "rb_gemm_bf16: internal: bad K split %d", parts);
  const long long tiles = (long long)m_tiles * n_tiles;
  RB_REQUIRE(tiles < (1LL << 30), "rb_gemm_bf16: too many tiles");
  // byte offsets inside a tile are 32-bit
  RB_REQUIRE((long long)(BN > BM ? BN : BM) * k * 2 < (1LL << 32), "rb_gemm_bf16: K=%d too long for this kernel", k);
  RB_REQUIRE(!WF || n % 16 == 0, "rb_gemm_bf16: fragment-major W needs N=%d to be a multiple of 16", n);
  const size_t lds = (size_t)2 * (BN + BM) * 64 * sizeof(bf16_t);
  auto kern = gemm_pingpong_kernel<BN, BM, EPI, TO, WF, 0, false, ACT>;
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    RB_REQUIRE(e == hipSuccess, "rb_gemm_bf16: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    configured = true;
  }
  kern<<<dim3((unsigned)((tiles + 7) / 8 * 8), (unsigned)parts), 512, lds, s>>>(x, w, (TO*)c, parts > 1 ? slabs : nullptr, m, n, k, m_tiles,
                                                                                n_tiles, k / 64 / parts, rows.first, act, GemmGroups{nullptr, nullptr, 1});
  return 0;
}

template <int BN, int BM, int EPI, typename TO, bool WF>
static int launch_pingpong_cfg(const bf16_t* x, const bf16_t* w, void* c, int m, int n, int k, RowRange rows, hipStream_t s, int parts,
                               float* slabs, const float* act) {
  RB_REQUIRE(act == nullptr || c != nullptr, "rb_gemm_bf16: internal: an activation or a gate's numbers go with an output");
  int rc;
  if constexpr (EPI == 0) {
    if (act != nullptr && parts == 1) return launch_pingpong_kernel<BN, BM, EPI, TO, WF, true>(x, w, c, m, n, k, rows, s, 1, nullptr, act);
    rc = launch_pingpong_kernel<BN, BM, EPI, TO, WF, false>(x, w, c, m, n, k, rows, s, parts, slabs, nullptr);
    if (!rc && parts > 1 && c != nullptr) {       // without c the caller adds the slabs up itself
      const size_t count = (size_t)m * n;
      gemm_sum_slabs_kernel<TO><<<(unsigned)((count + 255) / 256), 256, 0, s>>>(slabs, (TO*)c, parts, count, act);
    }
  } else {
    rc = launch_pingpong_kernel<BN, BM, EPI, TO, WF, false>(x, w, c, m, n, k, rows, s, parts, slabs, act);
  }
  return rc;
}


template <int BN, int BM, int WN, int WM, int P, int EPI, typename TO>
static int launch_tiled_cfg(const bf16_t* x, const bf16_t* w, void* c, int m, int n, int k, hipStream_t s,
                            const float* act = nullptr) {
  const int m_tiles = (m + BM - 1) / BM, n_tiles = (n + BN - 1) / BN;
  const long long tiles = (long long)m_tiles * n_tiles;
  RB_REQUIRE(tiles < (1LL << 30), "rb_gemm_bf16: too many tiles");
  const size_t lds = (size_t)2 * (BN + BM) * TG_LD * sizeof(bf16_t);
  const bool tail = k % TG_BK != 0;
  auto kern = tail ? gemm_tiled_kernel<BN, BM, WN, WM, P, EPI, true, TO>
                   : gemm_tiled_kernel<BN, BM, WN, WM, P, EPI, false, TO>;
  static bool configured[2] = {false, false};
  if (!configured[tail]) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    RB_REQUIRE(e == hipSuccess, "rb_gemm_bf16: cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
    configured[tail] = true;
  }
  const int grid = (int)((tiles + 7) / 8 * 8);
  kern<<<grid, 64 * (BN / WN) * (BM / WM), lds, s>>>(x, w, (TO*)c, m, n, k, m_tiles, n_tiles, EPI <= 1 ? act : nullptr);
  return 0;
}

// ------------------------------------------------------------------ which tiles, how many K slices
// The kernels are bound by what they pull from L2 and LDS (a 128 x 128 x 64 tile needs a byte per
// 64 flop, a 256 x 256 one half of that), so the largest tile that still gives every compute unit
// work wins, and where even the smallest tiles are too few, K is cut into slices over workgroups
// (grid.y): each slice writes its partial sums to its own [M, N] slab of a workspace, and
// gemm_sum_slabs_kernel (or the kernel that reads them) adds them up in a fixed order.
//   on the kernel whose waves take turns (gemm_pingpong.h; 8 waves):
//   cfg 4: 256 rows of W x 256 tokens      cfg 6: 192 x 256      cfg 9: 128 x 256      cfg 8: 256 x 128
//   cfg 11: 192 x 128, cfg 5: 128 x 128 (2 workgroups per compute unit)
//   on the kernel of gemm_dma.h, where a tile is too small for eight waves:
//   cfg 7: 128 x 64, 3 stages deep (2 per compute unit)      cfg 13: the same with K tiles of 128
//   cfg 10: 64 x 64, 4 stages deep (2 per compute unit)
//   cfg 1..3: tiles staged through registers, for K that is no multiple of 64 (more than 64 tokens)
// Without K slices a product of 128 tokens by 4096 rows ran on 32 of the 256 compute units and
// took as long as one of 768 tokens (K = 14336: 194 us; 41 us with 4 slices of 64-token tiles).
struct TilePlan {
  int cfg;        // 0: not for the kernels of this file
  int parts;      // K slices; more than 1 needs parts * M * N floats of workspace
  int rest = 0;   // where the rows are dealt to two launches (no K slices then): the tiles of the second,
  int split = 0;  // and its first row
};

static int g_tile_cfg = 0, g_tile_parts = 0;
extern "C" void rb_tune_tiles(int cfg, int parts) {       // experiments only; 0 = built-in choice; + 100 * (tiles of a second launch)
  g_tile_cfg = cfg;
  g_tile_parts = parts;
}

// The choice among the tiles that are loaded straight into LDS and the number of K slices is the least of an estimate
// of every candidate's time, a sum whose terms were fitted to measured products: for more than 64 tokens 13,400 times of 580 products (29
// sizes of W, K 512 to 14,336, at 65 to 8,192 tokens, every tile with 1 to 8 slices forced in turn, W rotated over copies beyond the
// caches, the sums of slices apart; `bench.py --planner-sweep` repeats such a sweep), for 17 to 64 tokens 96 of six shapes at 24 to 64.
//
//   time [us] = c0 + K tiles of a slice x (what the compute units' tiles cost per K tile)
//               + fixed x (tiles on the busiest compute unit) + w x MB of W
//               + out x MB of float32 outputs, slices among them, or gate x millions of gated pairs
//               + what adding up the slices takes
//
// A round is one tile on every compute unit (`per_unit` tiles where that many fit), and in K tiles
// of 64 it costs `full`; a product's w workgroups are full rounds and a last one of
// rem workgroups.  A last round is cheaper than a full one and the cheaper the emptier (the
// compute units that have work share the memory system with fewer): `last + per_fill x rem / units`,
// and for the tiles that fit twice, once every unit has one, `second + per_second x (rem - units) / units`.
// The machine enters through the number of compute units alone.  For more than 64 tokens the choice is 0.4 % above the best candidate in the
// mean, within 5 % of it in 570 of the 580 and 20 % above it at worst (72 tokens by 8,192 rows at K = 8192); fitted to two thirds of the sizes of W,
// 0.3 to 0.8 % for the other third.  For 17 to 64 tokens 0.8 %, within 5 % in 90 of the 96.
struct TileCost {
  int cfg, rows, tokens, bk, per_unit;
  float c0, full, last, per_fill, second, per_second, fixed, w, out, gate;
};
struct CostTable {
  float slab;       // 17 to 64 tokens: what a MB of slices costs, their sum included
  const TileCost* tiles;
  int n_tiles;
};
static const TileCost kCostMany[] = {
    {4, 256, 256, 64, 1, 2.838f, 1.303f, 0.7147f, 0.5014f, 0.f, 0.f, 6.819f, 0.03584f, 0.0974f, 0.05812f},
    {5, 128, 128, 64, 2, 3.569f, 0.8656f, 0.4617f, 0.07921f, 0.7067f, 0.1693f, 1.128f, 0.05974f, 0.1282f, 0.f},
    {6, 192, 256, 64, 1, 2.987f, 1.037f, 0.7484f, 0.2013f, 0.f, 0.f, 3.817f, 0.04315f, 0.1525f, 0.2065f},
    {7, 128, 64, 64, 2, 3.276f, 0.599f, 0.3345f, 0.02616f, 0.4611f, 0.1671f, 0.7892f, 0.08291f, 0.1237f, 1.662f},
    {8, 256, 128, 64, 1, 2.261f, 0.7886f, 0.6168f, 0.1378f, 0.f, 0.f, 4.84f, 0.05987f, 0.1094f, 0.f},
    {9, 128, 256, 64, 1, 2.529f, 0.7407f, 0.6354f, 0.0592f, 0.f, 0.f, 2.17f, 0.04335f, 0.2121f, 0.3667f},
    {10, 64, 64, 64, 2, 2.772f, 0.3846f, 0.2352f, 0.f, 0.3132f, 0.08173f, 0.5103f, 0.06921f, 0.1375f, 1.562f},
    {11, 192, 128, 64, 2, 4.905f, 1.237f, 0.5608f, 0.08948f, 0.9398f, 0.2723f, 0.8626f, 0.06783f, 0.1372f, 0.04604f},
    {13, 128, 64, 128, 1, 1.95f, 0.3657f, 0.3025f, 0.05767f, 0.f, 0.f, 2.889f, 0.06945f, 0.1094f, 2.212f}};
static const TileCost kCostFew[] = {{7, 128, 64, 64, 2, 5.522f, 1.2099f, 0.3352f, 0.2479f, 0.8967f, 0.3f, -0.4082f, 0.f, 0.f, 0.f},
                                    {10, 64, 64, 64, 2, 5.522f, 0.6268f, 0.191f, 0.1144f, 0.4995f, 0.1176f, -0.1f, 0.f, 0.f, 0.f},
                                    {13, 128, 64, 128, 1, 5.522f, 0.6506f, 0.3182f, 0.2568f, 0.f, 0.f, 0.2565f, 0.f, 0.f, 0.f}};
static const CostTable kMany = {0.f, kCostMany, 9};          // more than 64 tokens
static const CostTable kFew = {0.6852f, kCostFew, 3};        // 17 to 64 tokens

// What adding up the slices of a product of more than 64 tokens costs.  A launch of its own (gemm_sum_slabs_kernel) takes 2.1 us and its bytes, 0.19 us
// a MB it reads and 0.2 a MB it writes (2,133 pairs of times, with and without it).  A kernel that reads the terms anyway reads
// more of them: 0.3 us and 0.165 a MB (a norm behind the product, over one term and over 2 to 8, 1,578 times).  One price for both, 0.25 us a
// MB, cut products whose sum is a launch into slices that cost more than they gave: 700 tokens by 3,072 rows at K = 2048 20.0 -> 26.4 us.
// (The first price is never below the second one: what is not cut for a reader is not cut for itself.)
static double cost_of_slices(bool own_sum, int p, int m, int n) {
  const double mb = 4e-6 * m * n;
  return own_sum ? 2.1 + 0.19 * p * mb + 0.2 * mb : 0.3 + 0.165 * (p - 1) * mb;
}

// How many of W's rows the whole rounds of a tile take (0: there are none, or nothing is left).
static int whole_rounds(const TileCost& t, int m, int n) {
  const long long m_tiles = (m + t.tokens - 1) / t.tokens, slots = (long long)rb_compute_units() * t.per_unit;
  const int split = (int)(m_tiles * (n / t.rows) / slots * slots / m_tiles) * t.rows;
  return split < n ? split : 0;
}

// A product of more than 64 tokens may be two launches: as many whole rounds of a large tile as there are, and the rows behind them with
// a tile that takes less than the round that would not be full: 2,048 tokens by 28,672 rows are 3.5 rounds of 256 x 256, or 3 and one of
// 128 x 256 (362 -> 350 us); 3,781 tokens by 10,304 rows at K = 2048 151 -> 142; 3,000 by 22,016 gated, K = 4096, 423 -> 394.  Taken where the
// estimate is better by 3 %: of two launches it is up to 5 % too low (8,600 tokens by 4,096 rows at K = 11,008, 2 % better by the estimate: 586 -> 605).
// own_sum: a product cut into slices is added up by a launch of its own, and not by the kernel that reads it.
static TilePlan plan_by_cost(int m, int n, int k, int epilogue, bool own_sum) {
  const CostTable& table = m > 64 ? kMany : kFew;
  const long long units = rb_compute_units();
  const int kt = k / 64;
  auto cost_of = [&](const TileCost& t, int rows, int p) {
    const long long w = (long long)((rows + t.rows - 1) / t.rows) * ((m + t.tokens - 1) / t.tokens) * p, slots = units * t.per_unit;
    const long long rounds = w / slots, rem = w - rounds * slots;
    double per_k = rounds * t.full;
    if (rem > 0 && rem <= units) per_k += t.last + t.per_fill * ((double)rem / units);
    if (rem > units) per_k += t.second + t.per_second * ((double)(rem - units) / units);
    double cost = t.c0 + (double)kt / p * per_k + t.fixed * ((w + units - 1) / units) + t.w * (2e-6 * rows * k);
    if (epilogue) cost += t.gate * (1e-6 * m * rows);
    else cost += t.out * (4e-6 * p * m * rows);
    if (p > 1) cost += m > 64 ? cost_of_slices(own_sum, p, m, rows) : table.slab * (4e-6 * p * m * rows);
    return cost;
  };
  auto one = [&](int rows, int slices, double* least) {     // the best of all tiles in one launch
    TilePlan best = {0, 1};
    for (int i = 0; i < table.n_tiles; ++i) {
      const TileCost& t = table.tiles[i];
      if (k % t.bk != 0) continue;
      for (int p = 1; p <= slices; ++p) {
        if ((k / t.bk) % p != 0 || (p > 1 && kt / p < 4)) continue;
        const double cost = cost_of(t, rows, p);
        if (best.cfg == 0 || cost < *least) {
          best = {t.cfg, p};
          *least = cost;
        }
      }
    }
    return best;
  };
  double least = 0.0;
  TilePlan best = one(n, epilogue ? 1 : 8, &least);
  if (m <= 64) return best;
  double bound = 0.97 * least;
  for (int i = 0; i < table.n_tiles; ++i) {
    const TileCost& t = table.tiles[i];
    if (t.rows * t.tokens < 192 * 256 || k % t.bk != 0) continue;
    const int split = whole_rounds(t, m, n);
    if (split == 0) continue;
    double behind = 0.0;
    const TilePlan rest = one(n - split, 1, &behind);
    const double cost = cost_of(t, split, 1) + behind;
    if (cost < bound) {
      best = {t.cfg, 1, rest.cfg, split};
      bound = cost;
    }
  }
  return best;
}

static TilePlan plan_tiles(int m, int n, int k, int epilogue, bool own_sum) {
  const long long R = rb_compute_units();
  const bool dma = k % 64 == 0 && (long long)k * 512 < (1LL << 32);
  if (!dma) {
    if (m <= 64) return {0, 1};
    const long long t256 = (long long)((m + 255) / 256) * ((n + 255) / 256);
    const long long t256x128 = (long long)((m + 127) / 128) * ((n + 255) / 256);
    if (g_tile_cfg >= 1 && g_tile_cfg <= 3) return {g_tile_cfg, 1};
    return {t256 >= R * 5 / 8 ? 3 : (k >= 8192 && t256x128 >= R * 25 / 32 ? 2 : 1), 1};
  }
  if (m <= 16) return {0, 1};
  if (g_tile_cfg >= 4) {
    const int cfg = g_tile_cfg % 100, rest = g_tile_cfg / 100;
    if (rest > 0) {
      for (const TileCost& t : kCostMany)
        if (t.cfg == cfg && m > 64)
          if (const int split = whole_rounds(t, m, n)) return {cfg, 1, rest, split};
      return {cfg, 1};
    }
    const int p = (epilogue == 0 && g_tile_parts > 0 && (k / 64) % g_tile_parts == 0) ? g_tile_parts : 1;
    return {cfg, p};
  }
  return plan_by_cost(m, n, k, epilogue, own_sum);
}

template <int EPI, typename TO, bool WF>
static int launch_tiles(int cfg, const bf16_t* x, const bf16_t* w, void* c, float* workspace, int m, int n, int k, RowRange rows, hipStream_t s,
                        int p, const float* act) {
  switch (cfg) {
    case 4: return launch_pingpong_cfg<256, 256, EPI, TO, WF>(x, w, c, m, n, k, rows, s, p, workspace, act);
    case 6: return launch_pingpong_cfg<192, 256, EPI, TO, WF>(x, w, c, m, n, k, rows, s, p, workspace, act);
    case 9: return launch_pingpong_cfg<128, 256, EPI, TO, WF>(x, w, c, m, n, k, rows, s, p, workspace, act);
    case 8: return launch_pingpong_cfg<256, 128, EPI, TO, WF>(x, w, c, m, n, k, rows, s, p, workspace, act);
    case 11: return launch_pingpong_cfg<192, 128, EPI, TO, WF>(x, w, c, m, n, k, rows, s, p, workspace, act);
    case 5: return launch_pingpong_cfg<128, 128, EPI, TO, WF>(x, w, c, m, n, k, rows, s, p, workspace, act);
    case 7: return launch_dma_cfg<128, 64, 32, 64, 64, 3, EPI, TO, WF>(x, w, c, m, n, k, rows, s, p, workspace, act);
    case 10: return launch_dma_cfg<64, 64, 32, 32, 64, 4, EPI, TO, WF>(x, w, c, m, n, k, rows, s, p, workspace, act);
    case 13: return launch_dma_cfg<128, 64, 32, 64, 128, 3, EPI, TO, WF>(x, w, c, m, n, k, rows, s, p, workspace, act);
    default: break;
  }
  if constexpr (!WF) {
    switch (cfg) {
      case 3: return launch_tiled_cfg<256, 256, 128, 64, 2, EPI, TO>(x, w, c, m, n, k, s, act);
      case 2: return launch_tiled_cfg<256, 128, 128, 64, 2, EPI, TO>(x, w, c, m, n, k, s, act);
      default: return launch_tiled_cfg<128, 128, 64, 64, 2, EPI, TO>(x, w, c, m, n, k, s, act);
    }
  }
  RB_REQUIRE(false, "rb_gemm_bf16: internal: fragment-major W with K=%d, which the direct-to-LDS kernels do not take", k);
  return 1;
}

template <int EPI, typename TO, bool WF>
static int launch_planned(const bf16_t* x, const bf16_t* w, void* c, float* workspace, int m, int n, int k,
                          hipStream_t s, const float* act) {
  const TilePlan plan = plan_tiles(m, n, k, EPI, c != nullptr);
  RB_REQUIRE(plan.cfg != 0, "rb_gemm_bf16: internal: M=%d N=%d K=%d is not a product for the tiled kernels", m, n, k);
  RB_REQUIRE(plan.parts == 1 || workspace != nullptr, "rb_gemm_bf16: M=%d N=%d K=%d needs a workspace of %lld floats",
             m, n, k, (long long)plan.parts * m * n);
  const int p = plan.parts;
  const int rc = launch_tiles<EPI, TO, WF>(plan.cfg, x, w, c, workspace, m, n, k, {0, plan.rest ? plan.split : n}, s, p, act);
  if (rc || !plan.rest) return rc;
  return launch_tiles<EPI, TO, WF>(plan.rest, x, w, c, workspace, m, n, k, {plan.split, n}, s, 1, act);
}

#define RB_BY_OUTPUT(FN, WF, ...)                                                              \
  (epilogue == 0 ? (dtype_out == RB_F32 ? FN<0, float, WF>(__VA_ARGS__) : FN<0, bf16_t, WF>(__VA_ARGS__)) \
                 : (dtype_out == RB_F32 ? FN<1, float, WF>(__VA_ARGS__) : FN<1, bf16_t, WF>(__VA_ARGS__)))

// what the planner picks for these sizes, as 10000 * (the tiles of a second launch) + 100 * cfg + parts (0: not a product for this file)
extern "C" int rb_tune_plan(int m, int n, int k, int epilogue) {
  const TilePlan plan = plan_tiles(m, n, k, epilogue, true);
  return plan.cfg == 0 ? 0 : 10000 * plan.rest + 100 * plan.cfg + plan.parts;
}

int gemm_tiled_parts(int m, int n, int k, int epilogue, bool own_sum) {
  const TilePlan plan = plan_tiles(m, n, k, epilogue, own_sum);
  return plan.cfg == 0 ? 0 : plan.parts;
}

int gemm_tiled_launch(const bf16_t* x, const bf16_t* w, bool w_frag, void* c, float* workspace, int dtype_out,
                      int epilogue, int m, int n, int k, hipStream_t s, const float* act) {
  RB_REQUIRE(act == nullptr || epilogue <= 1, "rb_gemm_bf16: an activation goes with epilogue 0, a gate's numbers with epilogue 1");
  if (w_frag) return RB_BY_OUTPUT(launch_planned, true, x, w, c, workspace, m, n, k, s, act);
  return RB_BY_OUTPUT(launch_planned, false, x, w, c, workspace, m, n, k, s, act);
}
