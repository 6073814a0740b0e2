// The experts' weight gradients over few rows (gemm_outer.hip), as the expert GEMM entry points call them.
#pragma once
#include "common.hpp"

namespace pm {

struct OuterArgs {
    const void *A, *B;            // [batches][K][M], [batches][K][N], contiguous
    void *C;
    const int *live;              // [live_planes][batches]: rows in use, NULL: all
    int live_planes, live_round;
    int M, N, K, batches;
};

// whether it is the faster way; rows: expected of a batch
bool gemm_outer_serves(int dtype, int m, int n, int64_t k, int batches, int64_t rows);
int gemm_outer_run(int dtype, const OuterArgs &p, hipStream_t stream, const char *who);

} // namespace pm
