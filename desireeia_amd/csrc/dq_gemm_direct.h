// dq_gemm_direct.h - the few-token prefill GEMM (dq_gemm_direct.hip) and the
// activation layout it reads.
#pragma once

#include <type_traits>

#include "dq_common.h"

// Largest token count of the direct kernel.
constexpr size_t DQ_GEMM_DIRECT_TOK = 128;

// The quantized activation of the direct kernel, written by the quantizer of
// dq_gemm.hip into the GEMM workspace: a = [cols/256][8 slices][4 items]
// [tokens padded to 16][8 halfs] (slice c of item g holds the format's columns
// 256 sb + 64 g + 8 c .. +7), minp = the Q4_K block sums [cols/256][n_tok][8],
// inv = 1/s per token.
struct DqDirectAct {
    const _Float16* a;
    const _Float16* minp;
    const float* inv;
};

// Where the quantizer puts the direct layout of a format in a GEMM workspace.
DqDirectAct dq_gemm_direct_act(int fmt, size_t cols, size_t n_tok, void* work);

// Whether a product takes the direct kernel: up to DQ_GEMM_DIRECT_TOK tokens
// (half of it for more than 8192 rows, whose 128-token tiles of dq_gemm.hip
// already give 112 workgroups) of any shape whose bytes 32-bit offsets reach.
// With its quantizer against dq_gemm.hip's tiles, us at 29 / 64 / 128 tokens:
// Q6_K 4096 x 14336 29 / 37 / 46 against 91 / 93 / 101; Q8_0 4096 x 4096
// 13 / 16 / 21 against 53 / 56 / 60; Q4_K 14336 x 4096 24 / 30 / 47 against
// 35 / 39 / 45. Up to the limit a token's sum does not depend on the token
// count, so a prompt cut into chunks keeps its sums.
bool dq_gemm_direct_ok(int fmt, size_t rows, size_t cols, size_t n_tok);

// Up to DQ_GEMM_DIRECT_JOBS matrices with the same cols on activations of the
// same tokens: one launch per format, Q4_K and Q6_K together. tiled: w is the
// tile copy of dq_gemm_tiles_pack.
constexpr int DQ_GEMM_DIRECT_JOBS = 4;
struct DqDirectJob {
    int fmt;
    bool tiled;
    const void* w;
    size_t rows;
    DqDirectAct act;
    float* y;
};
int dq_gemm_direct(const DqDirectJob* jobs, int n, size_t cols, size_t n_tok, hipStream_t s);
