// naiwa_moe_decode calls of several rows, with the expert GEMMs on the matrix cores
// (decode_mfma.hip): segments and activations in one launch, gate/up per (64
// features, slot segment), down per (rows, K part, slot segment) into unweighted
// partial dots, and the ordered combine.
#pragma once

#include "common.h"

// Most pairs per token the combine orders.
#define NAIWA_MFMA_MAX_WIDTH 16

// Whether the call's formats and shapes fit the matrix-core decode.
bool naiwa_decode_mfma_ok(const naiwa_bank* gate, const naiwa_bank* up, const naiwa_bank* down, const void* x);

// Scratch of one pass over `rows` rows.
struct NaiwaMfmaLayout {
    size_t off_key, off_begin, off_perm, off_inv, off_ha, off_hs, off_he, off_xa, off_xs, off_xr, off_dpart, total;
    NaiwaMfmaLayout(int rows, int width, int H, int I, int kparts, int down_dtype);
};

// Rows per pass of a call in the fewest passes that fit `bytes` of scratch each (1 when none
// do).  A row's result does not depend on the rows beside it, so a call in several passes
// gives the bits of one pass.
extern "C" int naiwa_decode_mfma_rows_per_pass(int rows, int width, int H, int I, int kparts, int down_dtype,
                                               size_t bytes);

// Strips of 64 down rows a block of a call of `rows` rows of `width` pairs (decode_mfma.hip);
// exact_q4: Q4_K down weights, not rounded to bf16.
extern "C" int naiwa_decode_mfma_down_strips(int rows, int width, int slots, int H, int kparts, int exact_q4);

// One pass over scratch ws (NaiwaMfmaLayout(rows, ...).total bytes): out = (accumulate ? out
// : 0) + the weighted experts, and with res (bf16 [rows, H]) x = bf16(x + out) in place
// (out may then be null).  K parts of ks values of I, kparts of them.
// bf16: x, h and the weights are rounded to bf16 (a layer of a chain), otherwise the weights
// are exact.
int naiwa_decode_mfma(const naiwa_bank* gate, const naiwa_bank* up, const naiwa_bank* down, const void* x, int x_dtype,
                      const uint32_t* slot_ids, const float* w, int rows, int width, int act, float* out,
                      int accumulate, uint16_t* res, int ks, int kparts, bool bf16, uint8_t* ws, hipStream_t st);
