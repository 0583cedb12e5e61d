// Hooks for measurements and for tests that must reach a kernel the dispatcher would not pick.
// They are no part of the library's interface: nothing on the product path calls them, and
// only tests and measurement scripts bind them.  The settings are process-wide and are read at
// every launch; 0 restores the built-in choice.
#pragma once

#ifdef __cplusplus
extern "C" {
#endif

void rb_tune_compute_units(int n);                              // every planner: pretend the GPU has n compute units
void rb_tune(int rows_per_wave, int waves);                     // skinny product
void rb_tune_parts(int parts);                                  // skinny product: 1 or 2 workgroups for a tile of 16 rows
int rb_tune_few_parts(int m, int n, int k, int epilogue);       // the same: the built-in choice
int rb_tune_few_aside(int n, int k, int epilogue);              // skinny product of 9 to 16 tokens: whether operands are set aside
int rb_tune_few_blocks(int m, int n, int k, int epilogue, int prepared);      // skinny product: the built-in choice of blocks of depth a load of the tokens
int rb_tune_group_form(int m, int k, int tiles);                // products in one launch: the built-in choice of how the tokens are loaded
void rb_tune_resident(int tiles);                               // skinny product with resident tokens: row tiles per workgroup
void rb_tune_use_resident(int on);                              // 0: never the resident variant, 2: also below 8192 rows
void rb_tune_f32_few(int on);                                   // float32 product of few tokens: 0 = on the vector units, not the float32 MFMA; 3 = one row tile a wave always
void rb_tune_f32_parts(int parts);                              // the same: 1 or 2 workgroups for a tile of 16 rows
int rb_tune_f32_ahead(int m, int n);                            // the same: the built-in choice, 1 = a second stage in registers
void rb_tune_f32_tile(int tile);                                // float32 product of many tokens: 1..7 = that tile, -1 = tiles staged through registers
int rb_tune_f32_plan(int m, int n, int k);                      // float32 product of many tokens: the built-in choice, 10 * (tile of a second launch) + tile
int rb_tune_singles_by_seq(int n_seqs, int n_heads, int dim, int vdim);      // recurrences of single tokens: the built-in choice of their order
void rb_tune_use_stream(int on);                                // 0: the skinny product up to 64 tokens
void rb_tune_tiles(int cfg, int parts);                         // tiled product: tile configuration (+ 100 * that of a second launch) and K slices
int rb_tune_plan(int m, int n, int k, int epilogue);            // tiled product: the built-in choice, 10000 * (tiles of a second launch) + 100 * cfg + parts
void rb_tune_attention_vec(int on);                             // generic attention: 0 = the scalar kernel also for head sizes that are multiples of 4, 2 = the vector units for float32 too
void rb_tune_prefill_waves(int waves);                          // prefill attention: 4 or 8
void rb_tune_prefill_paired(int on);                           // prefill attention: 0 = late blocks first only, no pairing of heavy and light workgroups
void rb_tune_decode_mfma(int mode);                             // decode attention: 1 bfloat16 weights also for one query head per kv head
void rb_tune_decode_waves(int waves);                           // decode attention: 2 or 4 waves a workgroup

#ifdef __cplusplus
}
#endif
