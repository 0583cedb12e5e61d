// Launchers of the bfloat16 matrix-core products, one per source file; rb_gemm_bf16 picks
// among them.  Each returns 0, or an error code with the message stored.
#pragma once
#include <hip/hip_runtime.h>

#include "mfma.h"

// The token operand of a product: bfloat16 rows of K values; row i of the product is row
// rows[i] of x (row i without rows).  With squares ([*, ceil(K / 16)], rows as in x) the rows are
// a float32 row times a norm's gain and squares holds that float32 row's sums of squares, one
// for every 16 columns: the product is multiplied by 1 / sqrt(their sum / K + eps), which makes
// it the product of the RMS-normalised row.
struct GemmTokens {
  const bf16_t* x;
  const float* squares;
  float eps;
  const int32_t* rows;
};

// What becomes of the sums.  epilogue 0: C = sums; 1: the gated pair; 2: C (float32) += sums;
// 3: as 2, and for the norm that follows gained [M, N] = bf16(C * gain) and
// squares [M, ceil(N / 16)] = the sums of C^2 over every 16 columns.
//
// w_frag says how W [N, K] is stored.  false: rows of K values.  true: fragment-major, for K % 64
// == 0 and N % 16 == 0: blocks of 16 rows x 32 depth values, 1 KB each, in the order [N / 16][K / 32];
// inside a block the 16 bytes of lane l of an MFMA's row operand (row l % 16, depth values
// 8 (l / 16) .. + 7) lie at 16 l.  A wave's load instruction then reads 1 KB in a row, and a
// product of few tokens reads W once with non-temporal loads: 6.0-6.8 TB/s instead of 5.3-5.8.
struct GemmAfter {
  int epilogue;
  const float* gain;
  bf16_t* gained;
  float* squares;
  bool w_frag;
  const float* act = nullptr;      // epilogue 0: the two numbers of xIELU, applied to the sums before they are stored (null: none)
};

// An operand of at most 16 / XP rows (a product's tokens, or part of a tile of W), XP blocks of 32 depth values a load.  A wave-wide load costs its
// compute unit the same whether its lanes ask for different bytes or not, and a product of few tokens spent half of its loads on 16 columns of tokens
// most of which stand for none.  Lane r of 16 brings row r % (16 / XP) of block r / (16 / XP) instead, and a block's turn comes by a
// rotation inside the row of 16 lanes.  Rows behind the last then hold other blocks' numbers and their sums are dropped, as they always were; the others are the same
// bits.  us without and with, 1, 4 and 8 tokens: 2,048 rows at K = 8192 9.0 / 9.5 / 10.3 and 8.8 / 9.2 / 10.0, 10,304 at 2048 9.45 / 9.48 / 9.92 and 9.09 / 8.96 / 9.68,
// 4,096 at 14336 20.8 / 20.9 / 21.6 and 20.5 / 20.5 / 21.3.
template <int XP>
struct RowPack {
  static_assert(XP == 1 || XP == 2 || XP == 4, "a stage is four blocks");
  static __device__ __forceinline__ int row(int r) { return r % (16 / XP); }
  static __device__ __forceinline__ int depth(int r) { return 32 * (r / (16 / XP)); }
  // 16 bytes of block `turn` (a constant) of those that a load brought, in the lanes of the operand's rows
  template <typename V>
  static __device__ __forceinline__ V turned(const V& of, int turn) {
    static_assert(sizeof(V) == 16, "16 bytes a lane");
    if (XP == 1 || turn == 0) return of;
    struct Words {
      int v[4];
    };
    Words w = __builtin_bit_cast(Words, of);
#pragma unroll
    for (int i = 0; i < 4; ++i)                             // row_ror: lane r gets what lane (r - n) % 16 holds
      w.v[i] = 16 / XP * turn == 4   ? __builtin_amdgcn_update_dpp(w.v[i], w.v[i], 0x12C, 0xF, 0xF, true)
               : 16 / XP * turn == 8 ? __builtin_amdgcn_update_dpp(w.v[i], w.v[i], 0x128, 0xF, 0xF, true)
                                     : __builtin_amdgcn_update_dpp(w.v[i], w.v[i], 0x124, 0xF, 0xF, true);
    return __builtin_bit_cast(V, w);
  }
  // block j of those that these loads brought
  template <int N>
  static __device__ __forceinline__ Frag8 block(const Frag8 (&b)[N], int j) {
    Frag8 f;
    f.u = turned(b[j / XP].u, j % XP);
    return f;
  }
};

// A lane's share of a row's n_sq sums of squares: `share` of `shares` (4 lanes of every wave work
// on one row).  With n_sq a multiple of 4 the first 16 * shares * SQ_WIDE of them are asked for
// with 16-byte loads that are all in flight together, and added up by squares_sum() when they
// are needed; the rest, if any, one by one.
template <int SQ_WIDE = 4>
struct SquaresShare {
  float4 wide[SQ_WIDE];
  float rest;
};
template <int SQ_WIDE = 4>
__device__ __forceinline__ SquaresShare<SQ_WIDE> squares_ask(const float* __restrict__ sq, int n_sq, int share, int shares) {
  SquaresShare<SQ_WIDE> out;
  out.rest = 0.f;
  int done = 0;
  if (n_sq % 4 == 0) {
#pragma unroll
    for (int j = 0; j < SQ_WIDE; ++j) {
      const int at = 4 * (share + j * shares);
      out.wide[j] = at < n_sq ? *reinterpret_cast<const float4*>(sq + at) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    done = 4 * shares * SQ_WIDE;
  } else {
#pragma unroll
    for (int j = 0; j < SQ_WIDE; ++j) out.wide[j] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  for (int i = done + share; i < n_sq; i += shares) out.rest += sq[i];
  return out;
}
template <int SQ_WIDE>
__device__ __forceinline__ float squares_sum(const SquaresShare<SQ_WIDE>& s) {
  float t = s.rest;
#pragma unroll
  for (int j = 0; j < SQ_WIDE; ++j) t += (s.wide[j].x + s.wide[j].y) + (s.wide[j].z + s.wide[j].w);
  return t;
}

// at most 64 tokens, any K % 8 == 0: W streamed straight into MFMA operands (gemm_skinny.hip);
// prepared tokens and epilogues 2 and 3: at most 16 tokens
int gemm_skinny_launch(const GemmTokens& x, const bf16_t* w, void* c, int dtype_out, const GemmAfter& after, int m,
                       int n, int k, hipStream_t s);
// at most 16 tokens kept in registers while a workgroup walks several row tiles; false: these
// sizes are not for it and nothing was launched
bool gemm_resident_try(const GemmTokens& x, const bf16_t* w, void* c, int dtype_out, const GemmAfter& after, int m,
                       int n, int k, hipStream_t s, int* rc);
bool gemm_resident_takes(int m, int k, int parts);
// For several products in one launch (gemm_group.hip), K % 128 == 0: the waves that share K with one row tile a wave, and whether a product
// alone takes its sums in that order (the same waves, whatever row tiles each has, and not the kernel with resident tokens).
int gemm_skinny_waves(int n, int k);
bool gemm_skinny_waves_alone(int n, int k);
bool gemm_sums_alone_alike(int m, int n, int k);
// more than 16 tokens (more than 64 when K is no multiple of 64): tiles through LDS
// (gemm_tiled.hip).  gemm_tiled_parts: 0 when these sizes are not for it, else the number of K
// slices it will use; more than 1 needs parts * m * n floats of workspace.  own_sum: the slices are added up by a launch
// of the product's own, not by the kernel that reads them; a product that is one slice then is one for itself, too.
int gemm_tiled_parts(int m, int n, int k, int epilogue, bool own_sum);
int gemm_tiled_launch(const bf16_t* x, const bf16_t* w, bool w_frag, void* c, float* workspace, int dtype_out,
                      int epilogue, int m, int n, int k, hipStream_t s, const float* act = nullptr);
// float32, more than 16 tokens, K % 32 == 0: tiles through LDS on the float32 MFMA (gemm_f32.hip); false: these operands are not
// for it and nothing was launched
bool gemm_f32_dma_try(const float* x, const float* w, bool w_frag, float* c, int m, int n, int k, hipStream_t s, int* rc);
