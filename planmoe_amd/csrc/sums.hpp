// The last stage of the reductions whose first stage leaves sums in fp32: of shares of rows, or of a product's tiles.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pm {

// out[e][c] = the sum of from[e][slot][c] over the batch's slots.  live: a slot holds the sum of slot_rows / per_tile rows of the batch's
// rows in use, slots behind them hold nothing; NULL: all slots count.
struct SumJob {
    const float *from;
    void *out;
    int batches, slots, cols;
    const int *live;
    int live_planes, live_round, rows, slot_rows, per_tile;
};
constexpr int SUM_JOBS = 3;
// up to SUM_JOBS reductions in one launch, out in dtype
int sum_slots(const char *who, int dtype, const SumJob *jobs, int n, hipStream_t st);

// planmoe_expert_gemm_relu_bwd with other reductions' last stage in the launch of its own
int relu_bwd_with(const char *who, int dtype, const void *a, const void *b, const void *h, int batches, int m, int n, int k, const int *live,
                  int live_planes, int live_round, int rows_hint, void *c, void *dbias, void *workspace, size_t workspace_bytes,
                  const SumJob *others, int others_n, hipStream_t st);

} // namespace pm
