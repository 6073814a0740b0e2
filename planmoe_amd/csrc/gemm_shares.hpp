// A product of the experts (bf16, nn) whose sums are left in shares of the reduction for the launch that reads them next.
#pragma once
#include "gemm_skinny.hpp"

namespace pm {

struct GemmShares {
    int splits = 0;               // 0: the product is computed whole
    int active = 0;               // the most batches that have rows
    bool few = false;             // gemm_skinny.hip's kernel, else gemm_deep.hip's
};

// m, n, k: rows at most of a batch, columns, reduction; rows: expected of a batch; pairs: rows of all batches at most; most: shares at most
GemmShares gemm_shares_pick(int m, int n, int64_t k, int batches, int64_t rows, int64_t pairs, int64_t most);
// Whether they are the faster way, the combine's share of the work with them; coded: the combine takes the rows through the int8 codec
bool gemm_shares_pay(const GemmShares &how, int m, int n, int64_t k, int batches, int64_t rows, int64_t pairs, bool coded);
// p.shares, p.live and at most 64 batches; the caller has checked shape and alignment (as planmoe_expert_gemm does)
int gemm_shares_run(const GemmShares &how, SkinnyArgs p, hipStream_t stream, const char *who);
// what planmoe_expert_gemm refuses of its operands and their sizes
int expert_gemm_check(const char *who, int form, int dtype, const void *a, const void *b, int batches, int m, int n, int k,
                      const int32_t *live, int live_planes, int live_round, const void *c);

} // namespace pm
