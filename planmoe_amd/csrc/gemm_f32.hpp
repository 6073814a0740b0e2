// The fp32 product of the expert FFN as the expert GEMM entry points call it.
#pragma once
#include "common.hpp"

namespace pm {

struct Gemm32Args {
    const float *A, *B, *bias, *mask;      // mask: c is kept where mask > 0, else zero (relu's backward)
    float *C, *colsum;                     // colsum: [batches][2 tile rows][N] column sums of what was stored, NULL: none
    const int *live;                       // [live_planes][batches]: rows in use (k of a tn product), NULL: all
    int live_planes, live_round;
    int M, N, K, batches, relu;            // operands and result contiguous
};

// form: 0 nn, 1 nt, 2 tn; the caller has checked shape and alignment.  side: rows and columns of a tile, 64 or 128, or 0:
// no tiles, waves on their own (gemm_f32_tile picks it for a number of rows in use); column sums then have two slots for 64 rows
int gemm_f32_tile(int form, const Gemm32Args &p, int rows_hint);
int gemm_f32_run(int form, const Gemm32Args &p, int side, hipStream_t stream, const char *who);

} // namespace pm
