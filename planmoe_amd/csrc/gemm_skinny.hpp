// The experts' product for few rows, as the expert GEMM entry points call it.
#pragma once
#include "common.hpp"

namespace pm {

constexpr int SKINNY_ROWS = 32;                             // the most rows of an expert it takes

struct SkinnyArgs {
    const uint16_t *A, *B, *bias;
    const uint16_t *mask;         // relu's backward (nt): c is kept where mask > 0, NULL: none
    uint16_t *C;
    float *colsum;                // with mask: column sums of what was stored, [batches][N], NULL: none
    const int *live;              // [live_planes][batches]: rows in use, NULL: all
    int live_planes, live_round;
    int M, N, K, batches, relu;   // operands and result contiguous
    float *shares = nullptr;      // in place of C: fp32 sums over a share of k each, [splits][batches][M][N], without bias and relu
    int splits = 1, active = 0;   // (shares) how many; the most batches that have rows
};

// a weight that is read past the caches
bool skinny_large(int64_t n, int64_t k, int64_t batches);
// the columns that a work-group takes
int gemm_skinny_width(bool nt, int n, int64_t k, int batches);
// nt: b is [batches, N, K], else [batches, K, N]; the caller has checked shape and alignment
int gemm_skinny_run(bool nt, SkinnyArgs p, hipStream_t stream, const char *who);
// nn into shares, live given, at most 64 batches: work-groups of 64 columns for the batches that have rows
int gemm_skinny_shares_run(const SkinnyArgs &p, hipStream_t stream, const char *who);

} // namespace pm
