// The experts' product in few tiles, as the expert GEMM entry points call it.
#pragma once
#include "gemm_skinny.hpp"

namespace pm {

// whether the operands are within reach of a 32-bit offset from a tile's corner
bool gemm_deep_reaches(int form, int m, int n, int64_t k);
// columns: 128 or 64 of a tile; form: 0 nn, 1 nt, 2 tn (live: rows in use of k); with mask (nt): colsum has two slots for every 128 rows; the caller has checked shape and
// alignment
int gemm_deep_run(int form, int columns, const SkinnyArgs &p, hipStream_t stream, const char *who);
// nn into shares (SkinnyArgs): a work-group for a tile and a share of its k-tiles
int gemm_deep_shares_run(const SkinnyArgs &p, hipStream_t stream, const char *who);
constexpr int DEEP_BK = 64;       // k of a k-tile

} // namespace pm
