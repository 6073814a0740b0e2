// The fp32 product of the expert FFN as the expert GEMM entry points call it.
#pragma once
#include "common.hpp"

namespace pm {

struct Gemm32Args {
    const float *A, *B, *bias, *mask;      // mask: c is kept where mask > 0, else zero (relu's backward)
    float *C, *colsum;                     // colsum: [batches][2 tile rows][N] column sums of what was stored, NULL: none
    const int *live;                       // [live_planes][batches]: rows in use (k of a tn product), NULL: all
    int live_planes, live_round;
    int M, N, K, batches;                  // operands and result contiguous
    int relu;
};

// Kernels: waves on their own; tiles of 64 x 64 (two and four k-tiles in LDS), 32 x 32 (five, and eight), and 128 x 128 on the fp32 matrix cores; tiles of 64 x 64, 128 x 128 and 256 x 128
// on the bf16 matrix cores, the operands in three parts
enum Gemm32Kernel { G32_WAVES, G32_TILE_64, G32_DEEP_64, G32_SLIM, G32_SLIM_ALONE, G32_TILE_128, G32_SPLIT_64, G32_SPLIT_128, G32_SPLIT_256 };

// form: 0 nn, 1 nt, 2 tn; the caller has checked shape and alignment.  rows_hint: rows in use
Gemm32Kernel gemm_f32_pick(int form, const Gemm32Args &p, int rows_hint);
int gemm_f32_run(int form, const Gemm32Args &p, Gemm32Kernel kernel, int rows_hint, hipStream_t stream, const char *who);
int gemm_f32_slim_run(int form, bool alone, const Gemm32Args &p, hipStream_t stream, const char *who);        // nn, nt
int gemm_f32_split_run(int form, const Gemm32Args &p, Gemm32Kernel kernel, hipStream_t stream, const char *who);
// column sums have two slots for so many rows
inline int gemm_f32_slot_rows(Gemm32Kernel kernel) { return kernel == G32_TILE_128 || kernel == G32_SPLIT_128 || kernel == G32_SPLIT_256 ? 128 : 64; }

} // namespace pm
