// ah_few.h -- launch arguments of the few-token GEMM (ah_few.hip), planned by ah_abi.cpp.
#pragma once

#include "ah_internal.h"

constexpr uint32_t kFewMaxWaves = 16;
constexpr uint32_t kFewMaxParts = 4;

struct FewPart {
    const uint8_t *w;
    float *y;          // [n_tok][n_out]
    uint32_t w_bytes, row_bytes, n_out, wg_begin;
    uint64_t key0;     // added to the part's output refusal keys
};
struct FewArgs {
    FewPart p[kFewMaxParts];  // FFN: gate, up
    const void *x;            // f32 [n_tok][n_in], or int8 codes (rows `pitch` bytes apart) with `scales`
    const int64_t *scales;    // [n_tok][ceil(n_in / 32)] with AH_SRC_CODES
    unsigned long long *status;
    uint32_t n_parts, n_in, n_tok, kpad, src, pitch;
    uint32_t splits;          // waves along K of a row tile
    uint32_t waves;           // of a workgroup: splits x row tiles
    uint32_t tok_tile;        // tokens of a workgroup (<= 32)
    uint32_t tok_tiles, n_wg; // filled by ah_launch_few
    float *gy, *uy;           // FFN: f32 gate / up values, or nullptr
    int8_t *h_codes;          // FFN: [n_tok][n_ff]
    int64_t *h_scales;        // FFN: [n_tok][ceil(n_ff / 32)]
};
