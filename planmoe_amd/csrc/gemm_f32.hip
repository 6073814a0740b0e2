// Batched fp32 GEMM of the expert FFN (experts/ffn.py:63-82 and its backward pass) on gfx950's fp32 matrix
// cores (v_mfma_f32_32x32x2_f32: fp32 products and sums, 157 TFLOP/s):
//   C[e][m][n] = act( sum_k A[e][m][k] * B[e][n][k] + bias[e][n] )
// with either operand stored k fast or k slow, as planmoe_gemm_*_bf16.
//
// A 32 x 32 x 2 MFMA takes 64 clocks, so unlike bf16 nothing here is bound by operand traffic: a 128 x 128
// tile reads 32 KB per k-tile of 32 for 4096 clocks of matrix core.  Four waves of 64 x 64 (32 x 32 in the small
// tile), operands straight into LDS (buffer_load ... lds), the next k-tile in flight during the MFMAs of this one, two work-groups
// per compute unit so that one's barrier and epilogue fall under the other's MFMAs.  Where there are few tiles of 64 x 64 a wave is alone on its
// matrix core, and what it issues ahead of a k-tile's products (a barrier, descriptors, loads, LDS reads: 440 of 1600 clocks) is time lost: the
// form with four stages has one descriptor for a whole operand, places in LDS known when it is compiled, and puts every load and read
// between two products.  A k-fast operand is
// read four k at a time (16 bytes per lane), sixteen k are two reads, and the sums take them in the order
// 0 4 8 12, 1 5 9 13, ..: the order of a product made of 16 x 16 x 4 instructions whose lanes read 16 bytes, so what such
// a product (the fp32 library's) gives, this one gives bit for bit, and a relu behind it cuts the same elements.
// (Larger products that no such relu follows are gemm_f32_split.hip's.)
#include "gemm_f32_core.hpp"
#include <algorithm>
#include <cmath>
#include <type_traits>

namespace pm {

// F: 32 x 32 fragments of a wave on a side; the tile is 64 F x 64 F.  STAGES: k-tiles in LDS, two or four.  With four a wave reads the first
// fragments of the next k-tile beside the products of this one.  (us, cold weights, two and four stages: 4 experts x 256 rows, 1024 -> 512 25 and 19;
// 3072 -> 1024 72 and 56; 8 x 24, 2048 -> 2048 b^T 55 and 38.)
template <int F, bool TA, bool TB, int STAGES>
__global__ __launch_bounds__(256, 2) void gemm_f32_kernel(const Gemm32Args p)
{
    constexpr int G32_B = 64 * F, G32_OPERAND = G32_B * G32_BK * 4;         // tile side; one operand's k-tile in LDS (A0 A1 .. B0 B1 ..)
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;

    const int tiles_m = (p.M + G32_B - 1) / G32_B, tiles_n = (p.N + G32_B - 1) / G32_B;
    int e, m0, n0, M = p.M, K = p.K;
    if constexpr (TA) {                          // (the rows in use are the reduction's)
        const int total = tiles_m * tiles_n * p.batches, per_xcd = (total + 7) / 8;
        const int tile = blockIdx.x % 8 * per_xcd + blockIdx.x / 8;
        if (blockIdx.x / 8 >= per_xcd || tile >= total) return;
        e = tile / (tiles_m * tiles_n);
        int in = tile - e * tiles_m * tiles_n;
        const int panel = in / (tiles_m * 8);
        in -= panel * tiles_m * 8;
        const int width = min(8, tiles_n - panel * 8);
        m0 = in / width * G32_B;
        n0 = (panel * 8 + in % width) * G32_B;
        if (p.live) {
            int n = 0;
            for (int j = 0; j < p.live_planes; ++j) n += p.live[j * p.batches + e];
            K = min(K, (n + p.live_round - 1) / p.live_round * p.live_round);
        }
    } else {
        const G32Tile tile = g32_tile(p, G32_B, STAGES == 4 && F == 1 ? 32 : 0, tiles_n, 1);
        if (tile.e < 0) return;
        e = tile.e;
        m0 = tile.m * G32_B;
        n0 = tile.n * G32_B;
        M = tile.rows;
    }

    const int lda = TA ? p.M : p.K, ldb = TB ? p.N : p.K;
    const uint8_t *A = reinterpret_cast<const uint8_t *>(p.A + (int64_t)e * p.M * p.K + (TA ? (int64_t)m0 : (int64_t)m0 * lda));
    const uint8_t *B = reinterpret_cast<const uint8_t *>(p.B + (int64_t)e * p.N * p.K + (TB ? (int64_t)n0 : (int64_t)n0 * ldb));
    const int64_t ra = TA ? ((int64_t)(K - 1) * lda + (p.M - m0)) * 4 : ((int64_t)(M - m0 - 1) * lda + p.K) * 4;
    const int64_t rb = TB ? ((int64_t)(K - 1) * ldb + (p.N - n0)) * 4 : ((int64_t)(p.N - n0 - 1) * ldb + p.K) * 4;
    const int64_t step_a = TA ? (int64_t)G32_BK * lda * 4 : G32_BK * 4, step_b = TB ? (int64_t)G32_BK * ldb * 4 : G32_BK * 4;
    const int KT = __builtin_amdgcn_readfirstlane((K + G32_BK - 1) / G32_BK), k_tail = K % G32_BK ? K % G32_BK : G32_BK;

    // k fast: 64 F rows of 128 bytes, a load fills eight, chunk c of row r at unit c ^ (r >> 1) & 7.
    // k slow: 32 rows of 256 F bytes, a load fills 4 / F.
    auto fetch = [&](bool T, int i, int ld) -> uint32_t {
        if (T) return (uint32_t)(8 * wave + lane / (16 * F)) * (uint32_t)ld * 4u + (uint32_t)(lane % (16 * F)) * 16u;
        const int row = 16 * F * wave + 8 * i + (lane >> 3);
        return (uint32_t)row * (uint32_t)ld * 4u + (uint32_t)((lane & 7) ^ ((row >> 1) & 7)) * 16u;
    };
    const uint32_t va[2] = {fetch(TA, 0, lda), fetch(TA, TA ? 0 : 1, lda)}, vb[2] = {fetch(TB, 0, ldb), fetch(TB, TB ? 0 : 1, ldb)};
    // (chunks of a k-fast row past the end of K are asked for out of range)
    auto past = [&](int i) -> uint32_t { return (int)(((lane & 7) ^ ((4 * i + (lane >> 4)) & 7)) * 4) >= k_tail ? 0x80000000u : 0u; };
    const uint32_t past0 = past(0), past1 = past(1);
    // Four stages: the operands from their corner on are within reach of an offset (the caller sees to it), so a load is an offset away from
    // one descriptor and fits under a product; past the end the last k-tile is asked for again, so that the count of what is on its way stays
    // the same, and never used.
    const g32_u32x4 whole_a = g32_desc(A, ra), whole_b = g32_desc(B, rb);
    const int there = KT > 0 ? KT - 1 : 0;
    auto load = [&](int kt, int stage, int n) {  // the n-th of a k-tile's 4 F
        const bool last = kt == KT - 1 && k_tail != G32_BK, b = n >= 2 * F;
        const int i = b ? n - 2 * F : n;
        const bool T = b ? TB : TA;
        const uint32_t ld = (uint32_t)(b ? ldb : lda), v = (b ? vb[i & 1] : va[i & 1]) | (!T && last ? ((i & 1) ? past1 : past0) : 0u);
        const uint32_t rows = ld * 4u * (uint32_t)(T ? 4 / F * i : 8 * (i & ~1));
        const uint32_t to = lds0 + stage * G32_OPERAND + wave * (2048 * F) + (b ? STAGES * G32_OPERAND : 0) + i * 1024;
        if constexpr (STAGES == 4) {
            g32_dma16(b ? whole_b : whole_a, v, __builtin_amdgcn_readfirstlane(rows + (uint32_t)(kt < KT ? kt : there) * (uint32_t)(b ? step_b : step_a)), to);
        } else {
            g32_dma16(b ? g32_desc(B + kt * step_b, rb - kt * step_b) : g32_desc(A + kt * step_a, ra - kt * step_a), v, rows, to);
        }
    };
    auto load_tile = [&](int kt) {
        if (STAGES == 2 && kt >= KT) return;
#pragma unroll
        for (int n = 0; n < 4 * F; ++n) load(kt, kt & (STAGES - 1), n);
    };

    f32x16 acc[F][F];
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.f;
    const int fr = lane & 31, fc = lane >> 5;
    // sixteen k of a side's 32-row fragments: element q of half h of fragment i is k = 8 h + 4 fc + q
    auto read16 = [&](bool T, const uint8_t *base, int w, int s, f32x4 (&f)[F][2]) {
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (T) {
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        f[i][h][q] = *reinterpret_cast<const float *>(base + (16 * s + 8 * h + 4 * fc + q) * (256 * F) + (32 * F * w + 32 * i + fr) * 4);
                } else {
                    f[i][h] = *reinterpret_cast<const f32x4 *>(base + (32 * F * w + 32 * i + fr) * 128 + (((4 * s + 2 * h + fc) ^ ((fr >> 1) & 7)) * 16));
                }
            }
    };

    f32x4 fa[2][F][2], fb[2][F][2];
    auto read_a = [&](int stage, int s, int to) { read16(TA, lds + stage * G32_OPERAND, wm, s, fa[to]); };
    auto read_b = [&](int stage, int s, int to) { read16(TB, lds + (STAGES + stage) * G32_OPERAND, wn, s, fb[to]); };
    // (the second operand first: a lane then holds four consecutive columns of one row)
    auto multiply = [&](int s, int x) {
        const int q = x >> 1, h = x & 1;
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
            for (int j = 0; j < F; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[s][j][h][q], fa[s][i][h][q], acc[i][j], 0, 0, 0);
    };
#pragma unroll
    for (int kt = 0; kt < STAGES - 1; ++kt) load_tile(kt);
    // A tile of up to 32 rows, the last one of an expert as a rule: its waves take 16 columns each of all its rows, half (up to 16 rows a quarter) of the
    // time on the matrix cores that a wave with 32 rows of zeros beside the others takes.  A compute unit that has such a tile beside a whole one is what the
    // launch waits for.  16 x 16 x 4 with lane group g at k = 4 g + q: the sums have the same order.
    // us, 4 experts of 260, 250, 270 and 244 rows, 512 -> 1024, a pass of the product 21.9, so 17.3; b^T 21.3 and 16.2
    if constexpr (STAGES == 4 && F == 1 && !TA) {
        if (M - m0 <= 32) {
            const int l16 = lane & 15, g = lane >> 4, col = 16 * wave + l16;
            auto rows = [&](auto halves) {
                constexpr int H = decltype(halves)::value;        // 16 rows each
                f32x4 sum[H], a[2][H], b[2];
#pragma unroll
                for (int h = 0; h < H; ++h) sum[h] = f32x4{0.f, 0.f, 0.f, 0.f};
                auto read = [&](int stage, int s, int to) {
                    const uint8_t *at = lds + stage * G32_OPERAND, *bt = lds + (STAGES + stage) * G32_OPERAND;
#pragma unroll
                    for (int h = 0; h < H; ++h)
                        a[to][h] = *reinterpret_cast<const f32x4 *>(at + (16 * h + l16) * 128 + (((4 * s + g) ^ ((l16 >> 1) & 7)) * 16));
                    if (TB) {
#pragma unroll
                        for (int q = 0; q < 4; ++q) b[to][q] = *reinterpret_cast<const float *>(bt + (16 * s + 4 * g + q) * 256 + col * 4);
                    } else {
                        b[to] = *reinterpret_cast<const f32x4 *>(bt + col * 128 + (((4 * s + g) ^ ((l16 >> 1) & 7)) * 16));
                    }
                };
                auto products = [&](int from) {
#pragma unroll
                    for (int q = 0; q < 4; ++q)
#pragma unroll
                        for (int h = 0; h < H; ++h) sum[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[from][q], a[from][h][q], sum[h], 0, 0, 0);
                };
                asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"((STAGES - 2) * 4 * F) : "memory");
                read(0, 0, 0);
                for (int k0 = 0; k0 < KT; k0 += STAGES) {
#pragma unroll
                    for (int stage = 0; stage < STAGES; ++stage) {
                        const int kt = k0 + stage;
                        if (kt >= KT) break;
                        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((STAGES - 3) * 4 * F) : "memory");
                        __builtin_amdgcn_sched_barrier(0);
                        read(stage, 1, 1);
#pragma unroll
                        for (int n = 0; n < 4 * F; ++n) load(kt + STAGES - 1, (stage + STAGES - 1) % STAGES, n);
                        __builtin_amdgcn_sched_barrier(0);
                        products(0);
                        __builtin_amdgcn_sched_barrier(0);
                        read((stage + 1) % STAGES, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                        products(1);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                // a lane has columns 4 g .. + 3 of the wave's 16 of row l16
                const int n = n0 + 16 * wave + 4 * g;
                const bool in_n = n < p.N;                   // (N is a multiple of 4: a lane's columns are in or out together)
                float add[4], sums[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int x = 0; x < 4; ++x) add[x] = p.bias && in_n ? p.bias[(int64_t)e * p.N + n + x] : 0.f;
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    const int row = m0 + 16 * h + l16;
                    const int64_t to = ((int64_t)e * p.M + row) * p.N + n;
                    const bool inside = in_n && row < M;
                    f32x4 v = sum[h], keep = {0.f, 0.f, 0.f, 0.f};
                    float part[4];
                    if (p.mask && inside) keep = *reinterpret_cast<const f32x4 *>(p.mask + to);
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        if (p.bias) v[x] += add[x];
                        if (p.relu) v[x] = v[x] < 0.f ? 0.f : v[x];
                        if (p.mask) v[x] = keep[x] > 0.f ? v[x] : 0.f;
                        part[x] = inside ? v[x] : 0.f;
                    }
                    if (inside) *reinterpret_cast<f32x4 *>(p.C + to) = v;
                    if (p.colsum) {                          // (16 rows and 16 rows, as g32_store adds up the 32 of a wave)
#pragma unroll
                        for (int x = 0; x < 4; ++x) {
#pragma unroll
                            for (int d = 1; d < 16; d <<= 1) part[x] += __shfl_xor(part[x], d);
                            sums[x] += part[x];
                        }
                    }
                }
                if (p.colsum && l16 == 0 && in_n) {          // (two slots a tile; the second 32 rows are none)
                    float *to = p.colsum + ((int64_t)e * tiles_m * 2 + m0 / G32_B * 2) * p.N + n;
                    *reinterpret_cast<f32x4 *>(to) = f32x4{sums[0], sums[1], sums[2], sums[3]};
                    *reinterpret_cast<f32x4 *>(to + p.N) = f32x4{0.f, 0.f, 0.f, 0.f};
                }
            };
            if (M - m0 <= 16) rows(std::integral_constant<int, 1>{});
            else rows(std::integral_constant<int, 2>{});
            // nothing may still be on its way into LDS that another work-group gets
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            return;
        }
    }
    if constexpr (STAGES == 4) {
        // behind the barrier of k-tile kt everybody's share of kt + 1 is in as well, and everybody is done with kt - 1; what else there is to do
        // goes between the products, one thing at a time (ahead of them it left the matrix core idle for a third of a k-tile)
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"((STAGES - 2) * 4 * F) : "memory");
        read_a(0, 0, 0);
        read_b(0, 0, 0);
        for (int k0 = 0; k0 < KT; k0 += STAGES) {
#pragma unroll
            for (int stage = 0; stage < STAGES; ++stage) {       // (where things lie in LDS is known)
                const int kt = k0 + stage;
                if (kt >= KT) break;
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((STAGES - 3) * 4 * F) : "memory");
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int x = 0; x < 8; ++x) {
                    multiply(0, x);
                    __builtin_amdgcn_sched_barrier(0);
                    if (x == 0) read_a(stage, 1, 1);
                    else if (x == 1) read_b(stage, 1, 1);
                    else if (x - 2 < 4 * F) load(kt + STAGES - 1, (stage + STAGES - 1) % STAGES, x - 2);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int x = 0; x < 8; ++x) {
                    multiply(1, x);
                    __builtin_amdgcn_sched_barrier(0);
                    if (x == 0) read_a((stage + 1) % STAGES, 0, 0);
                    else if (x == 1) read_b((stage + 1) % STAGES, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    } else {
        for (int kt = 0; kt < KT; ++kt) {
            // this wave's share of k-tile kt is in; behind the barrier everybody's is, and everybody is done with kt - 1
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            load_tile(kt + 1);
            read_a(kt & 1, 0, 0);
            read_b(kt & 1, 0, 0);
            read_a(kt & 1, 1, 1);
            read_b(kt & 1, 1, 1);
#pragma unroll
            for (int x = 0; x < 16; ++x) multiply(x >> 3, x & 7);
        }
    }

    g32_store<F, F>(p, acc, e, m0, n0, M, wm, wn, m0 / G32_B * 2 + wm, tiles_m * 2);
    // nothing may still be on its way into LDS that another work-group gets
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Few rows: a wave on its own, 16 MF rows by 16 C columns, operands from memory straight into registers
// (no LDS, no barrier), 2 U steps of 16 k in flight.  v_mfma_f32_16x16x4_f32 with lane group g at k = 4 g + q: the sums
// take the k in the same order as the tiles do, so which kernel serves a shape does not show in the result.
// Bound by reading the weight, or, where a wave of 16 columns is all that a SIMD has, by what one wave has on its way (63 loads at most): nn reads
// a row of k at a time, 64 bytes with C = 1, a whole line with 2, 256 bytes with 4.  NT: past the caches.
template <int MF, int C, int U, bool TB, bool NT>
__global__ __launch_bounds__(256, 1) void gemm_f32_wave_kernel(const Gemm32Args p)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, g = lane >> 4;
    // The pieces of 16 MF rows by 64 columns that hold rows in use, batch by batch, the row blocks of a column next to each other
    // (they read the same weight); what is left of the grid has nothing to do.  (A grid over the capacity, with empty row
    // blocks between full ones, leaves whole groups of compute units with the empty ones, since work is handed to them in
    // turn: 64 experts of 32 rows, 4096 -> 1024, took 402 us at a capacity of 32 and 751 at 36, here 402 at both.)
    // Column sums have two slots for every 64 rows in use: the second of them may have no rows.
    auto blocks_of = [&](int rows) { return ((p.colsum ? (rows + 63) / 64 * 64 : rows) + 16 * MF - 1) / (16 * MF); };
    auto round_up = [&](int n) { return min(p.M, (n + p.live_round - 1) / p.live_round * p.live_round); };
    const int waves = blockDim.x >> 6, wide = 16 * C * waves, number = blockIdx.x, cols = (p.N + wide - 1) / wide, most = blocks_of(p.M);
    int e = number / (most * cols), M = p.M, blocks = most, piece = number - e * most * cols;
    if (p.live && most == 1) {                   // (a batch is a row block at most)
        int n = 0;
        for (int j = 0; j < p.live_planes; ++j) n += p.live[j * p.batches + e];
        M = round_up(n);
    } else if (p.live) {                         // (lane = batch)
        int n = 0;
        if (lane < p.batches)
            for (int j = 0; j < p.live_planes; ++j) n += p.live[j * p.batches + lane];
        const int rows = round_up(n);
        int ends = lane < p.batches ? blocks_of(rows) * cols : 0;
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(ends, d);
            if (lane >= d) ends += o;
        }
        if (number >= __builtin_amdgcn_readlane(ends, 63)) return;
        e = __builtin_amdgcn_readfirstlane(__popcll(__ballot(ends <= number)));        // (so many batches end before)
        M = __builtin_amdgcn_readlane(rows, e);
        blocks = blocks_of(M);
        piece = number - (e > 0 ? __builtin_amdgcn_readlane(ends, e - 1) : 0);
    }
    const int m0 = piece % blocks * 16 * MF, n0 = (piece / blocks * waves + wave) * 16 * C;
    if (M == 0 || n0 >= p.N) return;
    if (m0 >= M) {                               // (a second slot without rows)
        if (lane < 4 * C && n0 + 4 * lane < p.N)
            *reinterpret_cast<f32x4 *>(p.colsum + ((int64_t)e * ((p.M + 63) / 64 * 2) + m0 / 32) * p.N + n0 + 4 * lane) = f32x4{0.f, 0.f, 0.f, 0.f};
        return;
    }
    const float *A = p.A + (int64_t)e * p.M * p.K, *B = p.B + (int64_t)e * p.N * p.K;
    const __amdgpu_buffer_rsrc_t da = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(A), 0, M * p.K * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t db = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(B), 0, p.N * p.K * 4, 0x00020000);
    constexpr uint32_t NOWHERE = 0x80000000u;
    const int steps = (p.K + 15) / 16, col = n0 + C * l16;        // a lane's columns: C in a row, one in each fragment

    f32x4 acc[MF][C], fa[2][U][MF], fb[2][U][C];
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int c = 0; c < C; ++c) acc[m][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    // rows and columns past the end, and k past the end, read as zero
    auto load = [&](f32x4 (&a)[U][MF], f32x4 (&b)[U][C], int s0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = 16 * (s0 + u) + 4 * g;
            const bool in_k = k < p.K;
#pragma unroll
            for (int m = 0; m < MF; ++m) {
                const int row = m0 + 16 * m + l16;
                a[u][m] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(da, in_k && row < M ? ((uint32_t)row * (uint32_t)p.K + (uint32_t)k) * 4u : NOWHERE, 0, 0));
            }
            if (TB) {
                const uint32_t at = in_k && col < p.N ? ((uint32_t)k * (uint32_t)p.N + (uint32_t)col) * 4u : NOWHERE;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t row = (uint32_t)(q * 4) * (uint32_t)p.N;
                    if constexpr (C == 4) {
                        const pm_u32x4 v = __builtin_bit_cast(pm_u32x4, __builtin_amdgcn_raw_buffer_load_b128(db, at, row, NT ? 2 : 0));
#pragma unroll
                        for (int c = 0; c < 4; ++c) b[u][c][q] = __uint_as_float(v[c]);
                    } else if constexpr (C == 2) {
                        const pm_u32x2 v = __builtin_bit_cast(pm_u32x2, __builtin_amdgcn_raw_buffer_load_b64(db, at, row, NT ? 2 : 0));
                        b[u][0][q] = __uint_as_float(v[0]);
                        b[u][1][q] = __uint_as_float(v[1]);
                    } else {
                        b[u][0][q] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(db, at, row, NT ? 2 : 0));
                    }
                }
            } else {
#pragma unroll
                for (int c = 0; c < C; ++c)
                    b[u][c] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(db, in_k && col < p.N ? ((uint32_t)(col + c) * (uint32_t)p.K + (uint32_t)k) * 4u : NOWHERE, 0, NT ? 2 : 0));
            }
        }
    };
    // (the second operand first: a lane then holds four consecutive columns of one row)
    auto multiply = [&](const f32x4 (&a)[U][MF], const f32x4 (&b)[U][C]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int m = 0; m < MF; ++m)
#pragma unroll
                    for (int c = 0; c < C; ++c) acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[u][c][q], a[u][m][q], acc[m][c], 0, 0, 0);
    };
    load(fa[0], fb[0], 0);
    for (int s = 0; s < steps; s += 2 * U) {
        // (held in this order: moved behind the products to save registers, the loads would be waited for)
        load(fa[1], fb[1], s + U);
        __builtin_amdgcn_sched_barrier(0);
        multiply(fa[0], fb[0]);
        __builtin_amdgcn_sched_barrier(0);
        load(fa[0], fb[0], s + 2 * U);
        __builtin_amdgcn_sched_barrier(0);
        multiply(fa[1], fb[1]);
        __builtin_amdgcn_sched_barrier(0);
    }

    const int n = n0 + 4 * C * g;                // a lane's results: columns n .. n + 4 C - 1 of row l16, four in or out together
    float add[4 * C], sums[4 * C];
#pragma unroll
    for (int x = 0; x < 4 * C; ++x) {
        sums[x] = 0.f;
        add[x] = p.bias && n + x < p.N ? p.bias[(int64_t)e * p.N + n + x] : 0.f;
    }
#pragma unroll
    for (int m = 0; m < MF; ++m) {
        const int row = m0 + 16 * m + l16;
#pragma unroll
        for (int h = 0; h < C; ++h) {
            const int64_t at = ((int64_t)e * p.M + row) * p.N + n + 4 * h;
            const bool inside = n + 4 * h < p.N && row < M;
            f32x4 v, k = {0.f, 0.f, 0.f, 0.f};
            if (p.mask && inside) k = *reinterpret_cast<const f32x4 *>(p.mask + at);
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const int y = 4 * h + x;         // (column y: result y / C of fragment y % C)
                v[x] = acc[m][y % C][y / C];
                if (p.bias) v[x] += add[y];
                if (p.relu) v[x] = v[x] < 0.f ? 0.f : v[x];
                if (p.mask) { v[x] = k[x] > 0.f ? v[x] : 0.f; sums[y] += v[x]; }
            }
            if (inside) *reinterpret_cast<f32x4 *>(p.C + at) = v;
        }
    }
    if (p.colsum) {
#pragma unroll
        for (int x = 0; x < 4 * C; ++x)
#pragma unroll
            for (int d = 1; d < 16; d <<= 1) sums[x] += __shfl_xor(sums[x], d);
#pragma unroll
        for (int h = 0; h < C; ++h)
            if (l16 == 0 && n + 4 * h < p.N)
                *reinterpret_cast<f32x4 *>(p.colsum + ((int64_t)e * ((p.M + 63) / 64 * 2) + m0 / 32) * p.N + n + 4 * h) = f32x4{sums[4 * h], sums[4 * h + 1], sums[4 * h + 2], sums[4 * h + 3]};
    }
}

// weights that the last cache does not hold
static bool gemm_f32_past_caches(const Gemm32Args &p) { return (int64_t)p.batches * p.N * p.K * 4 > (int64_t)256 << 20; }
// pieces of 32 rows (16 where waves of 16 serve all of a batch's) by `columns` that the rows expected make
static int64_t gemm_f32_pieces(const Gemm32Args &p, int rows_hint, int columns)
{
    const int rows = p.M <= 16 && !p.colsum ? 16 : 32;
    return (int64_t)((rows_hint + rows - 1) / rows) * ((p.N + columns - 1) / columns) * p.batches;
}

// how many pieces of `rows` by `columns` the products have at most
static int64_t gemm_f32_wave_pieces(const Gemm32Args &p, int rows, int columns)
{
    const int64_t m = p.colsum ? ((int64_t)p.M + 63) / 64 * 64 : p.M;
    return (m + rows - 1) / rows * (((int64_t)p.N + columns - 1) / columns) * p.batches;
}

template <int MF, int C, int U, bool TB, bool NT = false>
static int gemm_f32_wave_launch(const Gemm32Args &p, int waves, hipStream_t stream, const char *who)
{
    gemm_f32_wave_kernel<MF, C, U, TB, NT><<<dim3((unsigned)gemm_f32_wave_pieces(p, 16 * MF, 16 * C * waves)), 64 * waves, 0, stream>>>(p);
    PM_LAUNCH_CHECK(who);
    return 0;
}

// Columns and waves of a work-group.  A wave reads whole lines with 32 columns, where there are such waves enough; 16 columns of short reductions;
// weights that the last cache (256 MB) does not hold go past the caches, 64 columns a wave.  b^T: a wave reads 64 bytes of every row whatever its columns.
// us with 16 columns and four waves a work-group everywhere, and now, weights cold, in the last cache:
//   8 x 1 row, 1024 -> 4096   33, 28 and 27, 22       8 x 7, 2600 -> 3440    80, 72 and 58, 52       16 x 512 -> 2048   20, 19 and 15, 14
//   8 x 20, 1024 -> 4096      44, 38 and 34, 28       16 x 1, 3328 -> 3072  149 and 95 (cold)
// (A row an expert by counts from the device, some of them without: single waves find a compute unit each, 16 x 224 -> 3136, 4 in use 11.0 and 8.5 us, all 14.1 and 13.0.)
static int gemm_f32_waves(int form, const Gemm32Args &p, int rows_hint, hipStream_t stream, const char *who)
{
    const int64_t strips = gemm_f32_pieces(p, rows_hint, 16), cu = compute_units();
    const bool one = p.M <= 16 && !p.colsum;
    if (form == 1) return one ? gemm_f32_wave_launch<1, 1, 4, false>(p, 1, stream, who) : gemm_f32_wave_launch<2, 1, 4, false>(p, 1, stream, who);
    if (strips < 4 * cu) return one ? gemm_f32_wave_launch<1, 1, 8, true>(p, 1, stream, who) : gemm_f32_wave_launch<2, 1, 4, true>(p, 1, stream, who);
    if (!one) return gemm_f32_wave_launch<2, 2, 4, true>(p, 1, stream, who);
    if (gemm_f32_past_caches(p) && strips >= 8 * cu) return gemm_f32_wave_launch<1, 4, 2, true, true>(p, 1, stream, who);
    return gemm_f32_wave_launch<1, 2, 4, true>(p, strips < 5 * cu || (p.live && rows_hint == 1) ? 1 : 4, stream, who);
}

template <int F, bool TA, bool TB, int STAGES = 2>
static int gemm_f32_launch(const Gemm32Args &p, hipStream_t stream, const char *who)
{
    constexpr int LDS = 2 * STAGES * 64 * F * G32_BK * 4, SIDE = 64 * F;
    const auto kernel = gemm_f32_kernel<F, TA, TB, STAGES>;
    static bool ready[64];                       // (per device; setting the attribute twice does no harm)
    int dev = 0;
    PM_REQUIRE(hipGetDevice(&dev) == hipSuccess, "%s: no device", who);
    if (dev >= 64 || !ready[dev]) {
        PM_REQUIRE(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) == hipSuccess,
                   "%s: the kernel needs %d bytes of LDS", who, LDS);
        if (dev < 64) ready[dev] = true;
    }
    const int64_t tiles = ((int64_t)p.M + SIDE - 1) / SIDE * (((int64_t)p.N + SIDE - 1) / SIDE) * p.batches;
    PM_REQUIRE(tiles < ((int64_t)1 << 30), "%s: too many tiles", who);
    kernel<<<dim3((unsigned)((tiles + 7) / 8 * 8 + (TA ? 0 : 8))), 256, LDS, stream>>>(p);
    PM_LAUNCH_CHECK(who);
    return 0;
}

// Four stages pay from eight k-tiles on (three are asked for before the first is multiplied), and need their operands within reach of an offset:
// 128 k past the end of one whose k is the slow index.
static bool gemm_f32_deep(int form, const Gemm32Args &p, int rows_hint)
{
    const int64_t reach = ((int64_t)1 << 31) / 4;
    if ((form == 2 ? rows_hint : p.K) <= 7 * G32_BK) return false;
    return (form == 1 || ((int64_t)p.K + 128) * p.N < reach) && (form != 2 || ((int64_t)p.K + 128) * p.M < reach);
}

// The tile's side under a relu: a compute unit takes 1.9 us for a k-tile of 128 x 128 and 4 for the tile, 0.52 and
// 1.2 for 64 x 64, 0.47 with four stages; what counts is the fullest compute unit (us, 64 x 64, with four stages, 128 x 128: 4 x 1000 rows,
// 2048 -> 512 77, 66, 137; 16 x 512, 1024 -> 1024 142, 131, 131; 512 -> 2048 152, 144, 138; 2 x 4096, 4096 -> 4096 2129, 1944, 1969).
// Up to 32 rows tiles of 32 x 32 (gemm_f32_slim.hip; five k-tiles in LDS, eight where that leaves work-groups room), or waves on their own: with fewer than
// eight k-tiles, where there is a wave of 32 columns for each SIMD and hardly a tile more than four for a compute unit to take in turn, for weights past the
// caches, and b^T with up to 16 rows where a compute unit has more than one tile and up to one and a half (up to two with up to 4 rows: a wave reads all rows for its 16
// columns): waves 0.86 - 0.94 of the tiles' time at any k, cold (8 x 3, 384 -> 1408 6.3 and 7.3, 4 x 14, 1180 -> 2176 14.8 and 15.8, 4 x 3, 3264 -> 2440 32 and 36).  us, weights cold, in the last cache, waves and tiles of 32 x 32:
//   nn  8 x 21 rows, 1896 -> 568  28, 28 and 16, 14      4 x 21, 2808 -> 1040  39, 39 and 19, 18      8 x 2, 4096 -> 1024    49, 37 and 27, 24
//       8 x 1, 1024 -> 4096       27, 23 and 34, 29      8 x 7, 3440 -> 2600   76, 66 and 65, 55      16 x 7, 1536 -> 2304   59, 51 and 51, 45
//       16 x 16, 1472 -> 2176     68, 60 and 49, 39      8 x 20, 1024 -> 4096  34, 27 and 38, 30      16 x 1, 2048 -> 2560   55, 55 and 70, 66
//   nt  8 x 21, 1896 -> 568       22, 22 and 14, 14      8 x 9, 2048 -> 2048   31, 27 and 31, 22      8 x 1, 1024 -> 4096    28, 23 and 32, 24
//       16 x 1, 3072 -> 3328      131 and 121            8 x 20, 1024 -> 4096  36, 29 and 33, 23
//   skewed, 8 experts, 128 of 256 rows on one, 4096 -> 1024 nn 67, 58 and 49, 40 (64 x 64 123)
// Beyond, tiles of 32 x 32 up to two a compute unit (eight k-tiles in LDS up to one), whose chains of products hide behind each other: a k-tile takes 0.275 us
// for both.  With more of them one takes 0.158 us each, a compute unit takes them in whole numbers, and 0.55 us each once; a k-tile of 64 x 64 takes 0.5 us, 1.5 of that
// beside a small one (several: 0.75 for each small one).  The weight costs 32 x 32 more, whose lines are asked for by more of them, and with its rows of k more
// still.  (Fitted to 2025 products of 33 to 400 rows, half of them within 5 %; what is picked is within 5 % of the faster one in 93 % of them.)  us, weights cold, tiles of 64 x 64
// and of 32 x 32:
//   nn  4 x 260 rows, 512 -> 1024  17, 19      1024 -> 512         22, 19      8 x 163, 2048 -> 256    36, 23      4 x 276, 1664 -> 2304   90, 91
//       8 x 66, 1024 -> 1024       22, 21      4 x 48, 3648 -> 1088 60, 34     8 x 100, 1024 -> 1024   23, 25      16 x 124, 3316 -> 768  115, 137
//       16 x 45, 1024 -> 256       20,  9      4 x 48, 1088 -> 3648 23, 26     16 x 97, 1536 -> 512    31, 34      8 x 288, 3200 -> 512   110, 91
//   nt  4 x 306, 972 -> 704        23, 24      8 x 178, 512 -> 512  14, 12     4 x 151, 2400 -> 2048   85, 70      4 x 330, 384 -> 1408    19, 21
// On the bf16 matrix cores, in three parts a value (gemm_f32_split.hip), where there is more than one tile of 64 x 64 for a compute
// unit; one tile on its own is bound by issuing the splits (8 experts, 128 rows, 1024 -> 1024: 20 us in fp32, 28 in parts) and stays here.
// A launch takes its rounds; us for a k-tile with few and with all compute units at work, and once for a tile, fitted to 60 shapes
// (within 7 %): in parts 64 x 64 0.6 alone, 0.44 each of several on a compute unit, + 6; 128 x 128 1.1 - 1.4, + 6; 256 x 128 1.9 - 2.5, + 7;
// in fp32 64 x 64 with four stages 0.43, 0.44 and + 4.
//   experts x rows, in, out       fp32 tiles    64     128    256 x 128
//   16 x 512, 1024, 1024 nn          147        126     102     88
//   16 x 512, 1024, 1024 tn          133        131     114     98
//   2 x 4096, 4096, 4096 nt         2005       1727    1434   1259
//   4 x 1000, 512, 2048 tn            75         66      52     76
//   8 x 300, 712, 712 nn              30         26      32     50
// Not under a relu, whose backward pass asks which elements it cut: one within rounding of zero that is cut here and kept there
// changes a weight gradient by 1e-3 of itself at 2^20 elements, so that product keeps the library's order of sums, and keeps it
// where no backward pass follows (a pass without autograd has the bits of the one with it: a checkpoint runs both).  Not up to
// 64 rows, where reading the weight takes as long as the fp32 matrix cores do (8 x 59, 3936 -> 3536: 136 us in fp32, 173 in parts).  And not
// with rows or columns of less than 256 values, where a product of few rows on waves has the same sums as one of many.
// Which of the two it is depends on the buffers' shape alone, not on the rows in use or expected: in parts the sums run in another
// order, and the layer as one node, which knows those rows, has to give the bits of its steps, which do not.  It is decided for all rows in use
// and for 4 of 5 (a capacity factor of 1.25), and only the tile by the rows expected.  Of 30000 products of layers with capacity factors of 1 to
// 1.5, 662 are computed in the slower way of the two for it, by 2.4 % on average by the figures above (for all rows alone 682, by 4.2 %).
// The far ends (us, 8 experts, fp32 and parts): capacity 72, 59 in use, 3936 -> 3536 136 and 173, all 72 in use 237 and 184; 952,
// 634 in use, 2240 -> 640 134 and 94.
struct SplitCost {                               // us: 64 x 64 in fp32; 64 x 64, 128 x 128, 256 x 128 in parts
    double whole, t64, t128, t256;
    double in_parts() const { return std::min(t64, std::min(t128, t256)); }
};

static SplitCost gemm_f32_split_cost(int form, const Gemm32Args &p, int64_t m, int64_t k)
{
    const double cu = compute_units(), kt = (double)((k + G32_BK - 1) / G32_BK);
    auto tiles = [&](int64_t bm, int64_t bn) { return (double)((m + bm - 1) / bm * ((p.N + bn - 1) / bn) * p.batches); };
    auto rounds = [&](double t, double low, double high, double once) {
        const double full = std::floor(t / cu), rest = t - full * cu;
        return full * (high * kt + once) + (rest > 0 ? (low + (high - low) * rest / cu) * kt + once : 0.);
    };
    const double small = std::ceil(tiles(64, 64) / cu), t64 = (small <= 1 ? 0.6 : 0.44 * small) * kt + 6;
    // (with two stages 0.52 a k-tile)
    const double whole = gemm_f32_deep(form, p, (int)k) ? (small <= 1 ? 0.43 : 0.44 * small) * kt + 3.5 + 0.5 * small : small <= 1 ? t64 : 1.18 * t64;
    return SplitCost{whole, t64, rounds(tiles(128, 128), 1.1, 1.4, 6), rounds(tiles(256, 128), 1.9, 2.5, 7)};
}

static bool gemm_f32_in_parts(int form, const Gemm32Args &p)
{
    if (p.relu || p.N < 256 || (form == 2 ? p.M : p.K) < 256) return false;
    const int64_t all = form == 2 ? p.K : p.M, most = (4 * all + 4) / 5;
    if (form != 2 && most <= 64) return false;
    auto cost = [&](int64_t rows) { return form == 2 ? gemm_f32_split_cost(form, p, p.M, rows) : gemm_f32_split_cost(form, p, rows, p.K); };
    const SplitCost a = cost(all), b = cost(most);
    return a.in_parts() * b.in_parts() < a.whole * b.whole;
}

Gemm32Kernel gemm_f32_pick(int form, const Gemm32Args &p, int rows_hint)
{
    if (gemm_f32_in_parts(form, p)) {
        // (row counts from the device: an expectation, and a batch may have a standard deviation more)
        const int64_t rows = p.live ? std::min<int64_t>(p.M, rows_hint + (int64_t)std::sqrt((double)rows_hint)) : rows_hint;
        const SplitCost c = gemm_f32_split_cost(form, p, form == 2 ? p.M : rows, form == 2 ? rows_hint : p.K);
        return c.t64 <= c.in_parts() ? G32_SPLIT_64 : c.t128 <= c.t256 ? G32_SPLIT_128 : G32_SPLIT_256;
    }
    const bool deep = gemm_f32_deep(form, p, rows_hint);
    const int64_t m = form == 2 ? p.M : rows_hint, cu = compute_units();
    const double kt = (double)(((form == 2 ? rows_hint : p.K) + G32_BK - 1) / G32_BK);
    if (form != 2 && rows_hint <= 32) {
        const int64_t pieces = gemm_f32_pieces(p, rows_hint, 32);
        // Rows for as many batches at most, by counts from the device: how many of those have one is not known, and waves of 32 and 64 columns that would fill the chip for all
        // are too few for a weight or three.  64 x 64, whose waves take 16 columns of up to 16 rows, is near the better one for any number.  us, waves and these, 16 experts, 2328 -> 3712:
        // 1 in use 50, 20   3 51, 22   8 58, 43   12 66, 83   16 82, 91;  8 experts, 2688 -> 4096: 1 55, 24   4 58, 36   8 59, 61;  512 -> 4096: 1 10.4, 7.9   4 13.4, 11.4   8 16.2, 18.7
        const bool some = p.live && rows_hint == 1 && deep;
        const bool one = p.M <= 16 && !p.colsum, past = gemm_f32_past_caches(p);
        const bool lines = pieces > 3 * cu && pieces <= 4 * cu && (one || (form == 0 && !past));
        const bool fits = (int64_t)p.M * p.K * 4 < ((int64_t)1 << 31) && (int64_t)p.N * p.K * 4 < ((int64_t)1 << 31) && gemm_f32_wave_pieces(p, 16, 16) < ((int64_t)1 << 30);
        if (some && form == 0 && (lines || (one && past && pieces >= 4 * cu))) return G32_DEEP_64;
        const bool turns = form == 1 && one && pieces > cu && 2 * pieces <= (rows_hint <= 4 ? 4 : 3) * cu;
        if (fits && (!deep || lines || turns || (form == 0 && one && past && pieces >= 4 * cu))) return G32_WAVES;
        if (deep) return pieces <= cu ? G32_SLIM_ALONE : G32_SLIM;
    }
    auto cost = [&](int64_t side, double us, double once) {
        const int64_t tiles = (m + side - 1) / side * ((p.N + side - 1) / side) * p.batches;
        return (double)((tiles + cu - 1) / cu) * (us * kt + once);
    };
    if (deep && form != 2) {
        // (row counts from the device: an expectation, and of many batches with a standard deviation of its root)
        double whole = 0, small = 0, slim = 0;
        for (const double q : {-1.5, -0.5, 0.5, 1.5}) {
            const int64_t r = p.live ? std::min<int64_t>(p.M, std::max<int64_t>(1, (int64_t)(m + q * std::sqrt((double)m)))) : m, rest = r % 64;
            whole += 0.25 * (double)(r / 64 + (rest > 32));
            small += 0.25 * (rest > 0 && rest <= 32);
            slim += 0.25 * (double)((r + 31) / 32);
        }
        const double columns = (double)((p.N + 63) / 64 * p.batches) / cu, mb = 4e-6 * (double)p.batches * p.N * p.K;
        whole *= columns;
        small *= columns;
        slim *= (double)((p.N + 31) / 32 * p.batches) / cu;
        const double us = kt * std::max(0.275, 0.158 * std::ceil(slim)) + 3.2 + 0.55 * slim + (form == 0 ? 0.065 : 0.027) * mb;
        const double deep_us = kt * 0.5 * (whole > 1 ? std::ceil(whole) + 0.75 * small : whole + small > 1 ? 1.46 : 1.) + 4.8 + 0.03 * mb;
        if ((slim <= 2 || us < deep_us) && us < cost(128, 1.9, 4)) return slim <= 1 ? G32_SLIM_ALONE : G32_SLIM;
    }
    return cost(64, deep ? 0.47 : 0.52, 1.2) < cost(128, 1.9, 4) ? deep ? G32_DEEP_64 : G32_TILE_64 : G32_TILE_128;
}

int gemm_f32_run(int form, const Gemm32Args &p, Gemm32Kernel kernel, int rows_hint, hipStream_t stream, const char *who)
{
    switch (kernel) {
    case G32_WAVES:
        return gemm_f32_waves(form, p, rows_hint, stream, who);
    case G32_TILE_64:
        if (form == 0) return gemm_f32_launch<1, false, true>(p, stream, who);
        if (form == 1) return gemm_f32_launch<1, false, false>(p, stream, who);
        return gemm_f32_launch<1, true, true>(p, stream, who);
    case G32_DEEP_64:
        if (form == 0) return gemm_f32_launch<1, false, true, 4>(p, stream, who);
        if (form == 1) return gemm_f32_launch<1, false, false, 4>(p, stream, who);
        return gemm_f32_launch<1, true, true, 4>(p, stream, who);
    case G32_SLIM: return gemm_f32_slim_run(form, false, p, stream, who);
    case G32_SLIM_ALONE: return gemm_f32_slim_run(form, true, p, stream, who);
    case G32_TILE_128:
        if (form == 0) return gemm_f32_launch<2, false, true>(p, stream, who);
        if (form == 1) return gemm_f32_launch<2, false, false>(p, stream, who);
        return gemm_f32_launch<2, true, true>(p, stream, who);
    default:
        return gemm_f32_split_run(form, p, kernel, stream, who);
    }
}

} // namespace pm
