// What the fp32 products' kernels share: buffer descriptors and a wave's results to memory.
#pragma once
#include "gemm_f32.hpp"

namespace pm {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t g32_u32x4 __attribute__((ext_vector_type(4)));

constexpr int G32_BK = 32;

__device__ __forceinline__ g32_u32x4 g32_desc(const void *base, int64_t bytes)
{
    const uint64_t a = (uint64_t)base;
    const uint32_t n = bytes <= 0 ? 0u : bytes > 0x7fffffff ? 0x7fffffffu : (uint32_t)bytes;
    return g32_u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, n, 0x00020000u};
}
__device__ __forceinline__ void g32_dma16(g32_u32x4 desc, uint32_t voff, uint32_t soff, uint32_t lds_addr)
{
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" :: "s"(lds_addr), "v"(voff), "s"(desc), "s"(soff) : "memory", "m0");
}

// sums over the lanes up to each: inside rows of 16, then the rows before
__device__ __forceinline__ int g32_prefix(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);         // row_shr 1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);        // row_bcast 15 into rows 1 and 3, 31 into rows 2 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
    return v;
}

// Where a work-group's tile lies.  XCD j (work-groups j, j + 8, ...) takes the j-th eighth of the tiles: batch, panel of 8 columns, row, column.  Only
// tiles that hold rows in use are dealt out, `step` rows of a batch at a time (the empty ones between them, in a grid over the capacity, fall on
// the same compute units again and again: 16 experts x 60 of 80 rows, 1024 -> 1024, 256 of 512 tiles of 64 x 64, 36 us, dealt out 24), and behind the others
// those of up to `small` rows, an eighth of them to each XCD as well (4 experts of 260, 250, 270 and 244 rows, 512 -> 1024, in one row with the others 22.6 us).
// The grid has eight work-groups more than there are tiles.
struct G32Tile { int e, m, n, rows; };           // rows in use of the batch; e < 0: there is no tile
__device__ __forceinline__ G32Tile g32_tile(const Gemm32Args &p, int bm, int small, int tiles_n, int step)
{
    const int lane = threadIdx.x & 63;
    auto rounded = [&](int rows) { return (rows + step - 1) / step * step; };
    auto whole_of = [&](int rows) { const int r = rounded(rows); return r / bm + (r % bm > small ? 1 : 0); };
    auto small_of = [&](int rows) { const int rest = rounded(rows) % bm; return rest > 0 && rest <= small ? 1 : 0; };
    int rows = p.M;
    if (p.live) {                                // (lane = batch)
        int n = 0;
        if (lane < p.batches)
            for (int j = 0; j < p.live_planes; ++j) n += p.live[j * p.batches + lane];
        rows = min(p.M, (n + p.live_round - 1) / p.live_round * p.live_round);
    }
    // (so many tiles up to the end of a batch; without row counts all batches are the same)
    auto ends_of = [&](int tiles) {
        if (!p.live) return __builtin_amdgcn_readfirstlane(tiles * tiles_n);
        return g32_prefix(lane < p.batches ? tiles * tiles_n : 0);
    };
    auto total_of = [&](int ends) { return __builtin_amdgcn_readfirstlane(p.live ? __builtin_amdgcn_readlane(ends, 63) : ends * p.batches); };
    G32Tile t{-1, 0, 0, p.M};
    int in = 0;
    auto find = [&](int ends, int number) {      // the batch of a tile, and its number there
        if (p.live) {
            t.e = __builtin_amdgcn_readfirstlane(__popcll(__ballot(ends <= number)));      // (so many batches end before)
            t.rows = __builtin_amdgcn_readlane(rows, t.e);
            in = number - (t.e > 0 ? __builtin_amdgcn_readlane(ends, t.e - 1) : 0);
        } else {
            t.e = __builtin_amdgcn_readfirstlane(number / ends);
            in = __builtin_amdgcn_readfirstlane(number - t.e * ends);
        }
    };
    const int xcd = blockIdx.x % 8, turn = blockIdx.x / 8, whole = ends_of(whole_of(rows)), wholes = total_of(whole), each = (wholes + 7) / 8;
    if (turn < each) {
        const int number = xcd * each + turn;
        if (number >= wholes) return t;
        find(whole, number);
        const int tiles_m = whole_of(t.rows), panel = in / (tiles_m * 8);
        in -= panel * tiles_m * 8;
        const int width = min(8, tiles_n - panel * 8);
        t.m = in / width;
        t.n = panel * 8 + in % width;
        return t;
    }
    if (small == 0) return t;
    const int part = ends_of(small_of(rows)), parts = total_of(part), number = xcd * ((parts + 7) / 8) + turn - each;
    if (turn - each >= (parts + 7) / 8 || number >= parts) return t;
    find(part, number);
    t.m = whole_of(t.rows);
    t.n = in;
    return t;
}

// A wave's 32 FM x 32 FN results at row 32 FM w_row, column 32 FN w_col of the tile at (m0, n0) of batch e: bias, relu, relu's
// backward, column sums into slot `slot` of `slots`.  Lane l holds row l % 32 of fragment i and of fragment j columns
// 8 q + 4 (l / 32) .. + 3 in acc[i][j][4 q ..]
template <int FM, int FN>
__device__ __forceinline__ void g32_store(const Gemm32Args &p, const f32x16 (&acc)[FM][FN], int e, int m0, int n0, int M, int w_row, int w_col,
                                          int slot, int slots)
{
    const int lane = threadIdx.x & 63, fr = lane & 31, fc = lane >> 5;
    const int64_t corner = (int64_t)e * p.M * p.N + (int64_t)m0 * p.N + n0;
    const int bytes = (int)min((int64_t)0x7fffffff, ((int64_t)(M - m0 - 1) * p.N + (p.N - n0)) * 4);
    const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(p.C + corner, 0, bytes, 0x00020000);
    float sums[FN][4][4];
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int col = w_col * 32 * FN + 32 * j + 8 * q + 4 * fc;
            const bool in_n = n0 + col < p.N;
            f32x4 add = {0.f, 0.f, 0.f, 0.f};
            if (p.bias && in_n) {
#pragma unroll
                for (int x = 0; x < 4; ++x) add[x] = p.bias[(int64_t)e * p.N + n0 + col + x];
            }
#pragma unroll
            for (int x = 0; x < 4; ++x) sums[j][q][x] = 0.f;
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                const int row = w_row * 32 * FM + 32 * i + fr;
                f32x4 v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
                if (p.bias) v += add;
                if (p.relu) {
#pragma unroll
                    for (int x = 0; x < 4; ++x) v[x] = v[x] < 0.f ? 0.f : v[x];
                }
                const bool inside = in_n && m0 + row < M;
                if (p.mask) {
                    f32x4 k = {0.f, 0.f, 0.f, 0.f};
                    if (inside) k = *reinterpret_cast<const f32x4 *>(p.mask + corner + (int64_t)row * p.N + col);
#pragma unroll
                    for (int x = 0; x < 4; ++x) { v[x] = k[x] > 0.f ? v[x] : 0.f; sums[j][q][x] += inside ? v[x] : 0.f; }
                }
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(pm_u32x4, v), out, in_n ? ((uint32_t)row * (uint32_t)p.N + (uint32_t)col) * 4u : 0x80000000u, 0, 0);
            }
        }
    if (p.colsum && slot < slots) {
        float *to = p.colsum + ((int64_t)e * slots + slot) * p.N + n0;
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
#pragma unroll
                for (int x = 0; x < 4; ++x)
#pragma unroll
                    for (int d = 1; d < 32; d <<= 1) sums[j][q][x] += __shfl_xor(sums[j][q][x], d);
                const int col = w_col * 32 * FN + 32 * j + 8 * q + 4 * fc;
                if (fr == 0 && n0 + col < p.N) *reinterpret_cast<float4 *>(to + col) = make_float4(sums[j][q][0], sums[j][q][1], sums[j][q][2], sums[j][q][3]);
            }
    }
}

} // namespace pm
