// dq_moe_tiles.h - the expert-tile weight layout (DQ_FMT_Q4_K_TILES) and the
// few-token expert FFN shared by dq_moe.hip and dq_moe_few.hip.
#pragma once

#include "dq_common.h"

// Expert tiles: per expert, tile of 128 rows and super-block a run of
// WT_BYTES, its 8 groups of 16 rows one after the other: for each two runs of
// 1 KB (16-byte slot (n, g), g = 0..3, n = 0..15 at (16 g + n) * 16: bytes 8g
// .. 8g+7 of the qs of items 2i and 2i + 1 of row n, i = 0, 1), then the 16
// super-block headers. Rows past the expert's end repeat its last row.
constexpr int WROWS = 128;
constexpr int WG_BYTES = 16 * 144;
constexpr int WT_BYTES = WROWS / 16 * WG_BYTES;

// The expert FFN of n_ent routed (token, slot) entries on int8 MFMA
// (dq_moe_few.hip): d_down [n_ent][n_embd] from the tokens x, the entries
// expert-major as pairs / offsets list them. work: dq_moe_few_bytes(n_ent).
// dq_moe_few: where it is the faster one, up to 12 entries per expert on
// average (an expert with more than 16 takes a second pass). Whole call,
// tiles, us against the 32-token fp16 kernel of dq_moe.hip, whose weight
// conversion serves all the tokens of a tile while the int8 kernel scales
// every token's partial sums: 8 experts top-2 of 4096 x 14336, 1 / 4 / 16 /
// 32 / 48 / 64 tokens 61 / 125 / 146 / 172 / 209 / 238 against 147 / 169 /
// 200 / 210 / 213 / 216; 32 experts top-4 of 2048 x 1024, 64 / 96 / 128
// tokens 66 / 75 / 99 against 79 / 90 / 99.
static inline bool dq_moe_few(uint32_t n_expert, size_t n_ent) { return n_ent <= 12 * (size_t)n_expert; }
size_t dq_moe_few_bytes(const dq_moe_t* m, size_t n_ent);
int dq_moe_few_ffn(const dq_moe_t* m, const float* d_x, const int32_t* d_pairs, const int32_t* d_offsets,
                   size_t n_ent, float** d_down, uint8_t* work, hipStream_t s);
