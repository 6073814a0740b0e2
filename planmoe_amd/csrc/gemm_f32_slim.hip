// The experts' fp32 product where there are few rows, or tiles of 64 x 64 are fewer than compute units: 32 x 32, fp32 matrix cores, nn and nt.
//
// Bound by reading the weight where there is much of it, else by the chain of a wave's products.  With 32 x 32 x 2 a wave takes 32 clocks for a k, whatever is
// idle beside it; here it has 16 x 16 of the result and takes 20 (a product of 16 x 16 x 4 waits some 80 clocks for the one before it: 64 x 32 tiles, two such
// chains a wave, take 740 clocks for a k-tile of 32, these 660), on four times the compute units, and the chains of the work-groups that share one
// hide behind each other.  Operands straight into LDS, five k-tiles, or eight where there are few work-groups and the trips to memory are what is waited for:
// 8 experts x 2 rows, 4096 -> 1024, cold, four, five and eight 47, 35, 27 us.  (Fragments read three steps ahead and no wait for them at the barrier: no gain.)
// 16 x 16 x 4 with lane group g at k = 4 g + q: the sums have the order of all the fp32 tiles, and the bits.
#include "gemm_f32_core.hpp"

namespace pm {

// Waves two by two, 16 rows by 16 columns each.  STAGES: k-tiles in LDS
template <bool TB, int STAGES>
__global__ __launch_bounds__(256, 4) void gemm_f32_slim_kernel(const Gemm32Args p)
{
    constexpr int OPERAND = 32 * 128;            // an operand's k-tile in LDS
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, l16 = lane & 15, g = lane >> 4;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;

    // (column sums have two slots for every 64 rows in use: the second of them may have no rows)
    const G32Tile tile = g32_tile(p, 32, 0, (p.N + 31) / 32, p.colsum ? 64 : 32);
    if (tile.e < 0) return;
    const int e = tile.e, m0 = tile.m * 32, n0 = tile.n * 32, K = p.K, M = tile.rows;
    // (a second slot without rows; multiplied like the others, 8 experts x 1 row, 768 -> 1536, 16.2 us, so 12.5; x 3, 920 -> 2184 24.6 and 18.5)
    if (m0 >= M) {
        if (tid < 8 && n0 + 4 * tid < p.N)
            *reinterpret_cast<f32x4 *>(p.colsum + ((int64_t)e * ((p.M + 63) / 64 * 2) + m0 / 32) * p.N + n0 + 4 * tid) = f32x4{0.f, 0.f, 0.f, 0.f};
        return;
    }

    const int ldb = TB ? p.N : p.K;
    const float *A = p.A + (int64_t)e * p.M * K + (int64_t)m0 * K, *B = p.B + (int64_t)e * p.N * K + (TB ? (int64_t)n0 : (int64_t)n0 * ldb);
    const g32_u32x4 da = g32_desc(A, ((int64_t)(M - m0 - 1) * K + K) * 4);
    const g32_u32x4 db = g32_desc(B, TB ? ((int64_t)(K - 1) * ldb + (p.N - n0)) * 4 : ((int64_t)(p.N - n0 - 1) * ldb + K) * 4);
    const int KT = __builtin_amdgcn_readfirstlane((K + G32_BK - 1) / G32_BK), last = KT - 1, k_tail = K % G32_BK ? K % G32_BK : G32_BK;

    // ---- rows of 128 bytes, a load fills eight.  k fast: chunk c of row r at unit c ^ (r >> 1) & 7.  k slow: row k at place k ^ (k >> 2 & 1), chunk c at
    // unit c ^ 4 (k >> 3 & 1), so that the four lane groups of a read, four k apart, lie in different quarters of the LDS's 256 bytes
    auto rows = [&](int row, int ld) -> uint32_t { return (uint32_t)row * (uint32_t)ld * 4u + (uint32_t)((lane & 7) ^ ((row >> 1) & 7)) * 16u; };
    const int place = 8 * wave + (lane >> 3), kb = place ^ ((place >> 2) & 1);
    const uint32_t va = rows(place, K), past = ((lane & 7) ^ ((place >> 1) & 7)) * 4 >= k_tail ? 0x80000000u : 0u;     // (chunks of a k-fast row past the end of K are asked for out of range)
    const uint32_t vb = TB ? (uint32_t)kb * (uint32_t)ldb * 4u + (uint32_t)((lane & 7) ^ (((kb >> 3) & 1) << 2)) * 16u : rows(place, ldb);
    const uint32_t step_b = TB ? (uint32_t)G32_BK * (uint32_t)ldb * 4u : G32_BK * 4u;
    // Past the end the last k-tile is asked for again, so that the count of what is on its way stays the same.
    auto load = [&](int kt, int stage) {
        const uint32_t end = kt == last && k_tail != G32_BK ? past : 0u, at = (uint32_t)min(kt, last), to = lds0 + stage * OPERAND + wave * 1024;
        g32_dma16(da, va | end, __builtin_amdgcn_readfirstlane(at * (G32_BK * 4u)), to);
        g32_dma16(db, vb | (TB ? 0u : end), __builtin_amdgcn_readfirstlane(at * step_b), to + STAGES * OPERAND);
    };

    f32x4 acc = {0.f, 0.f, 0.f, 0.f}, a[2], b[2];
    const int col = 16 * wn + l16;
    const uint8_t *to_a = lds + (16 * wm + l16) * 128, *to_b = lds + STAGES * OPERAND + (TB ? 0 : col * 128);
    auto read = [&](int stage, int s, int to) {  // sixteen k: lane group g has k = 16 s + 4 g + q
        const int unit = ((4 * s + g) ^ ((l16 >> 1) & 7)) * 16;
        a[to] = *reinterpret_cast<const f32x4 *>(to_a + stage * OPERAND + unit);
        if (TB) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                b[to][q] = *reinterpret_cast<const float *>(to_b + stage * OPERAND + (16 * s + 4 * g + (q ^ (g & 1))) * 128 + (((col >> 2) ^ ((g >> 1) << 2)) * 16) + (col & 3) * 4);
        } else {
            b[to] = *reinterpret_cast<const f32x4 *>(to_b + stage * OPERAND + unit);
        }
    };
    // (the second operand first: a lane then holds four consecutive columns of one row)
    auto multiply = [&](int from) {
#pragma unroll
        for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(b[from][q], a[from][q], acc, 0, 0, 0);
    };

#pragma unroll
    for (int kt = 0; kt < STAGES - 1; ++kt) load(kt, kt);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"((STAGES - 2) * 2) : "memory");
    read(0, 0, 0);
    for (int k0 = 0; k0 < KT; k0 += STAGES) {
#pragma unroll
        for (int stage = 0; stage < STAGES; ++stage) {
            const int kt = k0 + stage;
            if (kt >= KT) break;
            // behind the barrier everybody's share of k-tile kt + 1 is in as well, and everybody has read kt - 1
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((STAGES - 3) * 2) : "memory");
            __builtin_amdgcn_sched_barrier(0);
            read(stage, 1, 1);
            multiply(0);
            __builtin_amdgcn_sched_barrier(0);
            read((stage + 1) % STAGES, 0, 0);
            load(kt + STAGES - 1, (stage + STAGES - 1) % STAGES);
            multiply(1);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // ---- a lane has columns 4 g .. + 3 of the wave's 16 of rows l16
    const int n = n0 + 16 * wn + 4 * g;
    const bool in_n = n < p.N;                   // (N is a multiple of 4: a lane's columns are in or out together)
    const int row = m0 + 16 * wm + l16;
    const int64_t at = ((int64_t)e * p.M + row) * p.N + n;
    const bool inside = in_n && row < M;
    f32x4 v = acc, keep = {0.f, 0.f, 0.f, 0.f}, sums;
    if (p.mask && inside) keep = *reinterpret_cast<const f32x4 *>(p.mask + at);
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        if (p.bias && in_n) v[x] += p.bias[(int64_t)e * p.N + n + x];
        if (p.relu) v[x] = v[x] < 0.f ? 0.f : v[x];
        if (p.mask) v[x] = keep[x] > 0.f ? v[x] : 0.f;
        sums[x] = inside ? v[x] : 0.f;
    }
    if (inside) *reinterpret_cast<f32x4 *>(p.C + at) = v;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // nothing may still be on its way into LDS that another work-group gets
    if (p.colsum) {
        // 16 rows and 16 rows, as g32_store adds up the 32 of a slot
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int d = 1; d < 16; d <<= 1) sums[x] += __shfl_xor(sums[x], d);
        f32x4 *meet = reinterpret_cast<f32x4 *>(lds) + wn * 4 + g;
        __syncthreads();
        if (wm == 1 && l16 == 0) *meet = sums;
        __syncthreads();
        if (wm == 0 && l16 == 0 && in_n) *reinterpret_cast<f32x4 *>(p.colsum + ((int64_t)e * ((p.M + 63) / 64 * 2) + m0 / 32) * p.N + n) = sums + *meet;
    }
}

template <bool TB, int STAGES>
static int slim_launch(const Gemm32Args &p, hipStream_t stream, const char *who)
{
    constexpr int LDS = STAGES * 2 * 32 * 128;
    const auto kernel = gemm_f32_slim_kernel<TB, STAGES>;
    static bool ready[64];                       // (per device; setting the attribute twice does no harm)
    int dev = 0;
    PM_REQUIRE(hipGetDevice(&dev) == hipSuccess, "%s: no device", who);
    if (dev >= 64 || !ready[dev]) {
        PM_REQUIRE(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS) == hipSuccess,
                   "%s: the kernel needs %d bytes of LDS", who, LDS);
        if (dev < 64) ready[dev] = true;
    }
    const int64_t m = p.colsum ? ((int64_t)p.M + 63) / 64 * 64 : p.M, tiles = (m + 31) / 32 * (((int64_t)p.N + 31) / 32) * p.batches;
    PM_REQUIRE(tiles < ((int64_t)1 << 30), "%s: too many tiles", who);
    kernel<<<dim3((unsigned)((tiles + 7) / 8 * 8 + 8)), 256, LDS, stream>>>(p);
    PM_LAUNCH_CHECK(who);
    return 0;
}

int gemm_f32_slim_run(int form, bool alone, const Gemm32Args &p, hipStream_t stream, const char *who)
{
    if (form == 0) return alone ? slim_launch<true, 8>(p, stream, who) : slim_launch<true, 5>(p, stream, who);
    return alone ? slim_launch<false, 8>(p, stream, who) : slim_launch<false, 5>(p, stream, who);
}

} // namespace pm
