// Batched bf16 GEMM of the expert FFN, written for gfx950's matrix cores, and the transpose of its operands.
//
//   C[e][m][n] = act( bf16( bf16( sum_k A[e][m][k] * B[e][n][k] ) + bias[e][n] ) )
//
// A matrix-core operand is eight consecutive k per lane.  An operand stored with k running fastest
// ("N" for A, "T" for B) gives that as one 16-byte read of LDS; an operand stored the other way round
// is read through LDS reads that transpose (ds_read_b64_tr_b16), so the kernel takes either operand
// either way.  The reference's experts (experts/ffn.py:63-82) compute x @ fc1_w -> activation -> @ fc2_w
// with weights stored [experts, in, out]; the GEMM shapes of its forward and backward pass are
//   forward   y  = x  @ W          A = x  [rows, in],   B = W  [in, out]      planmoe_gemm_nn_bf16
//   backward  dx = dy @ W^T        A = dy [rows, out],  B = W  [in, out]      planmoe_gemm_nt_bf16
//             dW = x^T @ dy        A = x  [rows, in],   B = dy [rows, out]    planmoe_gemm_tn_bf16
// all with the operands as they lie in memory.
#include "gemm_f32.hpp"
#include "gemm_deep.hpp"
#include "gemm_outer.hpp"
#include "gemm_shares.hpp"
#include "sums.hpp"
#include <algorithm>
#include <cmath>

namespace pm {

typedef float  f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 gemm_bf16x8 __attribute__((ext_vector_type(8)));
typedef short gemm_s16x4 __attribute__((ext_vector_type(4)));
typedef short gemm_s16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t gemm_u32x4 __attribute__((ext_vector_type(4)));
typedef const uint8_t __attribute__((address_space(3))) *gemm_lds_ptr;

// ds_read_b64_tr_b16 hands lane i of every 16 lanes element i % 4 of the 8 bytes that lanes i / 4, i / 4 + 4, i / 4 + 8,
// i / 4 + 12 point at: with lane s pointing at row s / 4, columns 4 (s % 4) .. + 3 of a 4 x 16 patch, lane i receives 4
// consecutive k of column i -- the matrix cores' operand layout.  Two such reads make the 8 k of a step.
__device__ __forceinline__ gemm_bf16x8 gemm_read_tr(gemm_lds_ptr lo, gemm_lds_ptr hi)
{
    typedef gemm_s16x4 __attribute__((address_space(3))) *lds_s16x4;
    const gemm_s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)lo);
    const gemm_s16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)hi);
    return __builtin_bit_cast(gemm_bf16x8, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
}

// ---------------------------------------------------------------- the kernel
// Tiles of 256 x 256 (128 x 128; 128, 160 or 192 x 256), k-tiles of 64, four waves, two by two (or side by side, each with
// all rows).  Each side of a tile is two halves; a wave has 32 I rows of an A half and 32 J columns of either B half, so
// its share of the tile is four quadrants and a k-tile is four phases, one quadrant each: 4 I J v_mfma_f32_32x32x16_bf16.
// During a phase the wave reads from LDS the one half of an operand that the next phase needs and has
// not got (the quadrants of successive k-tiles are walked so that this is always one half), and asks
// for one half of a k-tile two further on, straight into LDS (buffer_load ... lds), into the space
// that the phase before has finished reading.  So a half is asked for seven phases (about 3500 clocks
// at 256 x 256) before it is read, LDS holds two k-tiles, and a phase ends in one wait -- by count, for
// the half the next phase reads -- and one barrier.  The loads and LDS reads are placed between the
// MFMAs one at a time: a wave issues in order, and a burst of them would leave its matrix core idle.
//
// The stream of k-tiles does not stop at the end of an output tile: work-groups stay (one per compute
// unit) and go from tile to tile, and the loads of the next tile's first k-tiles are in flight while
// the results of this one are rounded and stored.
//
// Out of range is the buffer descriptor's business: rows past the end, reduction rows past the end and
// everything behind the last tile read as zero, stores past the end are dropped.
//
// What bounds it: with operands of zeros 8 x 5120 x 4096 x 4096 takes 740 us (1860 TFLOP/s, 0.74 of the
// 2.5 PFLOP/s), with N(0, 1) operands 1030 - 1130 us (1220 - 1340): the clock the GPU holds under the
// matrix cores.  (A kernel with the same tile that waited for a whole k-tile at a time and issued its
// loads and LDS reads in bursts took 1260 us, 890 us with zeros.)
constexpr int GEMM_BK = 64;
constexpr int GEMM_WG = 256;
constexpr int GEMM_TABLE_BYTES = 2 * 64 * 4;                // tiles before each batch, its rows (with `live`)
constexpr int GEMM_BIAS_BYTES = 2 * 1024;                   // the tile's slice of the bias, two tiles in turn

struct GemmArgs {
    const uint16_t *A, *B, *bias;
    const uint16_t *mask;         // GRAD: c is kept where mask > 0 (c's shape and pitches), else zero
    uint16_t *C;
    float *colsum;                // GRAD: [batches][slots][N] column sums of what was stored, NULL: none; a slot for 128 rows and wave row (one wave row: a tile)
    const int *live;              // [live_planes][batches]: rows in use per batch (k of a tn product), NULL: all
    int live_planes, live_round;
    int M, N, K;
    int lda, ldb, ldc;            // elements between rows
    int64_t sA, sB, sC;           // elements between batches
    int batches, relu;
    int split;                    // 0: all tiles; 1: all but the last round's (gemm_last_round); 2: those, as quarters
    int stay;                     // work-groups of the 256 x 256 launch
    bool bias_by_value;           // the bias is not 16-byte aligned: read where it is used
};

__device__ __forceinline__ gemm_u32x4 gemm_desc(const void *base, int64_t bytes)
{
    const uint64_t a = (uint64_t)base;
    const uint32_t n = bytes <= 0 ? 0u : bytes > 0x7fffffff ? 0x7fffffffu : (uint32_t)bytes;
    return gemm_u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, n, 0x00020000u};
}
// how many of the 256 x 256 tiles, on work-groups that stay, would be left for a last round that is at most half full
__host__ __device__ inline int gemm_last_round(int tiles, int stay)
{
    const int last = tiles % stay;
    return 2 * last <= stay ? last : 0;
}
constexpr uint32_t GEMM_NOWHERE = 0x80000000u;              // an offset that is out of any descriptor's range
// 16 bytes per lane from the buffer at voff + soff to LDS at lds_addr + 16 * lane
__device__ __forceinline__ void gemm_dma16(gemm_u32x4 desc, uint32_t voff, uint32_t soff, uint32_t lds_addr)
{
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" :: "s"(lds_addr), "v"(voff), "s"(desc), "s"(soff) : "memory", "m0");
}
template <int N> __device__ __forceinline__ void gemm_phase_wait()
{
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory");
}

// WM x 4 / WM waves; in the halves of A a wave has I0 and I1 fragments of 32 rows, in those of B J fragments each of 32 columns
template <int WM_, int I0, int I1, int J_>
struct GemmShape {
    static constexpr int WM = WM_, WN = 4 / WM_, J = J_;
    static constexpr int I(int h) { return h ? I1 : I0; }
    static constexpr int IMAX = I0 > I1 ? I0 : I1;
    static constexpr int BM = 32 * WM * (I0 + I1), BN = 64 * WN * J;
    static constexpr int half(int o, int h) { return o == 0 ? 32 * WM * I(h) : 32 * WN * J; }        // rows (columns) of a half
    // LDS: both stages of A, both stages of B (so that an operand's halves are all within the 64 KB that an
    // LDS instruction's offset covers), the waves' output pieces (32 rows of 32 J values each), tables
    static constexpr int half_at(int o, int stage, int h)
    {
        return o == 0 ? stage * BM * 128 + h * half(0, 0) * 128 : 2 * BM * 128 + (2 * stage + h) * half(1, 0) * 128;
    }
    static constexpr int OPERANDS = 256 * (BM + BN);
    static constexpr int PITCH = 64 * J + 16;               // bytes between rows of an output piece
    static constexpr int TABLE = OPERANDS + 4 * 32 * PITCH, BIAS = TABLE + GEMM_TABLE_BYTES;
    static constexpr int LDS = BIAS + GEMM_BIAS_BYTES;
    static constexpr int STORES = 2 * (I0 + I1) * 2 * J;    // 16-byte stores of a lane per tile
    // loads a wave issues in phase p (the halves B B A1 A0), and how many of them may be outstanding at its end: the half that
    // phase p + 1 reads was asked for six phases before p, what is younger is not needed yet.  One wave row reads
    // the first pieces of A1 a phase ahead of the others (EARLY of them, with A's fragments read by all four waves a
    // phase would otherwise have more LDS reads than the products of a phase cover), so that half is there a phase earlier.
    static constexpr int EARLY = WM == 1 ? 4 * (I1 - 2) : 0;
    static constexpr int half_loads(int o, int h) { return half(o, h) / 32; }
    static constexpr int loads(int p) { return (p & 3) < 2 ? half_loads(1, 0) : half_loads(0, (p & 3) == 2); }
    static constexpr int wait(int p)
    {
        int s = 0;
        for (int j = 0; j < (EARLY > 0 && (p & 3) == 3 ? 5 : 6); ++j) s += loads(p - j + 8);
        return s;
    }
    static_assert(wait(3) + STORES < 64 && wait(1) + STORES < 64, "the counter of outstanding loads and stores has six bits");
    static constexpr int WAVES_PER_SIMD = LDS * 2 <= 160 * 1024 ? 2 : 1;     // (= work-groups per compute unit)
};
typedef GemmShape<2, 2, 2, 2> Gemm256;        // 256 x 256
typedef GemmShape<2, 1, 1, 1> Gemm128;        // 128 x 128
template <int I0, int I1> using GemmFlat = GemmShape<1, I0, I1, 1>;        // 32 (I0 + I1) x 256

template <class S, bool TA, bool TB, bool GRAD>
__global__ __launch_bounds__(GEMM_WG, S::WAVES_PER_SIMD) void gemm_bf16_kernel(const GemmArgs p)
{
    constexpr int J = S::J;
    static_assert(!TA || S::WM == 2, "a k-slow A: two wave rows");
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / S::WN, wn = wave % S::WN;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;

    // ---- the tiles: work-groups go to the 8 XCDs in turn, each XCD (with an L2 of its own) takes an
    // eighth of the tiles in a row, in the order batch, panel of 8 tile columns, tile row, column, so
    // that the tiles it works on at a time share operands (12 operand tiles for 32 products at 256 x 256).
    // With `live` the tiles of a batch are those of its rows in use: table[e] is the number before batch e.
    const int side = p.split == 2 ? 256 : S::BM, side_n = p.split == 2 ? 256 : S::BN;        // (of the tiles that are counted)
    const int tiles_n = (p.N + side_n - 1) / side_n;
    int total, base = 0;
    int *table = reinterpret_cast<int *>(lds + S::TABLE);
    if (p.live) {
        int n = 0;
        if (lane < p.batches)
            for (int j = 0; j < p.live_planes; ++j) n += p.live[j * p.batches + lane];
        const int rows = min(TA ? p.K : p.M, (n + p.live_round - 1) / p.live_round * p.live_round);
        const int mine = lane < p.batches ? ((TA ? p.M : rows) + side - 1) / side * tiles_n : 0;
        int inc = mine;
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(inc, d);
            if (lane >= d) inc += o;
        }
        // (every wave writes the same values and reads only what it wrote itself)
        table[lane] = lane < p.batches ? inc - mine : 0x7fffffff;
        table[64 + lane] = rows;
        total = __builtin_amdgcn_readlane(inc, 63);
    } else {
        total = (p.M + side - 1) / side * tiles_n * p.batches;
    }
    if (p.split == 1) total -= gemm_last_round(total, p.stay);
    if (p.split == 2) {
        const int last = gemm_last_round(total, p.stay);
        base = total - last;
        total = 4 * last;
    }
    const int per_xcd = (total + 7) / 8;
    const int first_tile = blockIdx.x % 8 * per_xcd, stride = gridDim.x / 8;
    struct Where { int e, m0, n0, rows; };        // rows: M of the batch (its K for a tn product)
    auto locate = [&](int j) {                    // j-th tile of this XCD (in range)
        const int number = first_tile + j, tile = p.split == 2 ? base + number / 4 : number;
        Where w;
        int first, tm;
        if (p.live) {
            // (batches without tiles share the next one's number: the last of them is the one)
            const int before = table[lane], rows = table[64 + lane];
            w.e = __builtin_amdgcn_readfirstlane(__popcll(__ballot(before <= tile)) - 1);
            first = __builtin_amdgcn_readlane(before, w.e);
            w.rows = __builtin_amdgcn_readlane(rows, w.e);
            tm = ((TA ? p.M : w.rows) + side - 1) / side;
        } else {
            tm = (p.M + side - 1) / side;
            w.e = tile / (tm * tiles_n);
            first = w.e * tm * tiles_n;
            w.rows = TA ? p.K : p.M;
        }
        int in = tile - first;
        const int panel = in / (tm * 8);
        in -= panel * tm * 8;
        const int width = min(8, tiles_n - panel * 8);
        w.m0 = in / width * side + (p.split == 2 ? (number & 2) * 64 : 0);
        w.n0 = (panel * 8 + in % width) * side_n + (p.split == 2 ? (number & 1) * 128 : 0);
        return w;
    };
    auto in_range = [&](int j) { return j < per_xcd && first_tile + j < total; };

    // ---- where the loads are: a cursor over the k-tiles of this work-group's tiles, one after another.
    // A tile takes an even number of k-tiles (the loop below does two at a time); the odd one past the end reads as zero.
    struct Cursor { const uint8_t *a, *b; int64_t ra, rb; int left, real, j; };    // left: k-tiles of the tile, real: without the padding
    const int64_t step_a = TA ? (int64_t)GEMM_BK * p.lda * 2 : GEMM_BK * 2, step_b = TB ? (int64_t)GEMM_BK * p.ldb * 2 : GEMM_BK * 2;
    auto k_of = [&](const Where &w) { return TA ? w.rows : p.K; };
    auto pairs = [](int K) { return max(1, (K + 2 * GEMM_BK - 1) / (2 * GEMM_BK)); };
    auto seek = [&](Cursor &c) {                  // to the first k-tile of tile c.j
        if (!in_range(c.j)) { c.ra = c.rb = 0; c.left = c.real = 0x7fffffff; return; }
        const Where w = locate(c.j);
        const int K = k_of(w), M = TA ? p.M : w.rows;
        c.a = reinterpret_cast<const uint8_t *>(p.A + w.e * p.sA + (TA ? (int64_t)w.m0 : (int64_t)w.m0 * p.lda));
        c.b = reinterpret_cast<const uint8_t *>(p.B + w.e * p.sB + (TB ? (int64_t)w.n0 : (int64_t)w.n0 * p.ldb));
        c.ra = TA ? ((int64_t)(K - 1) * p.lda + (M - w.m0)) * 2 : ((int64_t)(M - w.m0 - 1) * p.lda + K) * 2;
        c.rb = TB ? ((int64_t)(K - 1) * p.ldb + (p.N - w.n0)) * 2 : ((int64_t)(p.N - w.n0 - 1) * p.ldb + K) * 2;
        c.real = (K + GEMM_BK - 1) / GEMM_BK;
        c.left = pairs(K) * 2;
        if (K <= 0) c.ra = c.rb = 0;
    };
    auto advance = [&](Cursor &c) {
        if (--c.left == 0) { c.j += stride; seek(c); return; }
        c.a += step_a; c.b += step_b; c.ra -= step_a; c.rb -= step_b;
        if (--c.real <= 0) c.ra = c.rb = 0;
    };

    // ---- which 16 bytes of a half a lane fetches.  k fast: rows of 128 bytes, a load fills eight of
    // them, chunk c of row r lies at unit c ^ (r >> 1) & 7 (the 16 rows that one pass of a fragment read
    // touches then lie two by two in the halves of the LDS's 256 bytes, at eight different units).  k slow:
    // 64 rows of 128 X bytes (64 X rows or columns a half), chunk c of row k at unit c ^ (k & 3) << 2 (128-byte rows:
    // c ^ (k >> 1 & 1) << 2), so that the 4 rows of a transposing read's patch lie in different quarters of the 256 bytes.
    // Load i of a half: k fast, rows 8 i on (the swizzle turns with the parity of i); k slow, rows 8 / X i on.
    auto fetch = [&](bool T, int half, int i, int ld) -> uint32_t {
        if (T) {
            const int X = half / 64, kr = 16 * wave + lane / (8 * X), u = lane % (8 * X);
            return (uint32_t)kr * (uint32_t)ld * 2u + (uint32_t)(X == 2 ? u ^ ((kr & 3) << 2) : u ^ (((kr >> 1) & 1) << 2)) * 16u;
        }
        const int row = half / 4 * wave + 8 * i + (lane >> 3);
        return (uint32_t)row * (uint32_t)ld * 2u + (uint32_t)((lane & 7) ^ ((row >> 1) & 7)) * 16u;
    };
    uint32_t va[2][2], vb[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) { va[h][0] = fetch(TA, S::half(0, h), 0, p.lda); va[h][1] = TA ? va[h][0] : fetch(TA, S::half(0, h), 1, p.lda); }
    vb[0] = fetch(TB, S::half(1, 0), 0, p.ldb); vb[1] = TB ? vb[0] : fetch(TB, S::half(1, 0), 1, p.ldb);
    // a reduction length that is no multiple of 64: the chunks of a k-fast row past its end are asked for
    // out of range in a tile's last k-tile.  Chunk of a lane in load i: (lane & 7) ^ (4 (n + i) + (lane >> 4) & 7), n the
    // eights of rows of the half that lie before this wave's
    const int k_tail = TA || p.K % GEMM_BK == 0 ? GEMM_BK : p.K % GEMM_BK;      // (tn: both operands are k-slow)
    auto past = [&](int i) -> uint32_t {
        return (int)(((lane & 7) ^ ((4 * i + (lane >> 4)) & 7)) * 8) >= k_tail ? GEMM_NOWHERE : 0u;
    };
    const uint32_t past0 = past(0), past1 = past(1);      // (n + i even, odd)
    auto load = [&](int stage, int o, int h, int i, const Cursor &c) {
        const int half = S::half(o, h), each = S::half_loads(o, h), X = half / 64;
        const bool T = o == 0 ? TA : TB;
        const uint32_t dst = lds0 + S::half_at(o, stage, h) + wave * (each * 1024) + i * 1024;
        const uint32_t ld = (uint32_t)(o == 0 ? p.lda : p.ldb), first = h ? (uint32_t)S::half(o, 0) : 0u;
        const uint32_t soff = T ? ld * 2u * (uint32_t)(8 / (X > 0 ? X : 1) * i) + first * 2u : ld * 2u * ((uint32_t)(8 * (i & ~1)) + first);
        uint32_t v = o == 0 ? va[h][i & 1] : vb[i & 1];
        if (!T && k_tail != GEMM_BK) v |= c.real == 1 ? (((each & wave) + i) & 1 ? past1 : past0) : 0u;
        gemm_dma16(o == 0 ? gemm_desc(c.a, c.ra) : gemm_desc(c.b, c.rb), v, soff, dst);
    };

    // ---- fragments: 32 rows (columns) x 16 k; lane = row l % 32, k-chunk l / 32.  Where a lane's piece of the
    // first fragment of a half lies: k fast, one place for each of the four steps (the swizzle); k slow, one
    // for each fragment of the half
    gemm_bf16x8 fa[2][S::IMAX][4], fb[2][J][4];
    const int fr = lane & 31, fc = lane >> 5, tg = lane >> 4, ts = lane & 15;
    uint32_t ra[2][4], rb[4];                     // (A: by half, where the waves' shares differ)
    auto place = [&](bool T, int X, int share, int n, int w) -> uint32_t {        // share: fragments of a wave in the half
        if (T) {
            // lane = (group of 16 lanes, s): k row 8 (g / 2) + s / 4 of the step's 16, 8 bytes s % 4 of the 32 that columns
            // 16 (g % 2) .. + 15 of the fragment take
            const int row = 8 * (tg >> 1) + (ts >> 2), c = 4 * share * w + 4 * n + 2 * (tg & 1) + ((ts & 3) >> 1);
            const int u = X == 2 ? c ^ ((ts >> 2) << 2) : c ^ ((ts >> 3) << 2);
            return row * (128 * X) + u * 16 + 8 * (ts & 1);
        }
        return (32 * share * w + fr) * 128 + (((2 * n + fc) ^ ((fr >> 1) & 7)) * 16);
    };
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int n = 0; n < (TA ? S::I(h) : 4); ++n) ra[h][n] = lds0 + place(TA, S::half(0, h) / 64, S::I(h), n, wm);
#pragma unroll
    for (int n = 0; n < (TB ? J : 4); ++n) rb[n] = lds0 + S::half_at(1, 0, 0) + place(TB, S::half(1, 0) / 64, J, n, wn);
    auto read = [&](int stage, int o, int h, int r) {
        const int share = o == 0 ? S::I(h) : J, X = S::half(o, h) / 64, ks = r / share, i = r % share;
        const uint32_t at = (uint32_t)(S::half_at(o, stage, h) - S::half_at(o, 0, 0));
        gemm_bf16x8 f;
        if (o == 0 ? TA : TB) {
            const gemm_lds_ptr q = (gemm_lds_ptr)(uintptr_t)(o == 0 ? ra[h][i] : rb[i]) + at + ks * (16 * 128 * X);
            f = gemm_read_tr(q, q + 4 * 128 * X);
        } else {
            f = *(const gemm_bf16x8 __attribute__((address_space(3))) *)((gemm_lds_ptr)(uintptr_t)(o == 0 ? ra[h][ks] : rb[ks]) + at + i * 4096);
        }
        if (o == 0) fa[h][i][ks] = f; else fb[h][i][ks] = f;
    };

    f32x16 acc[2][2][S::IMAX][J];
    int fresh = 0;                                // the stores of the tile before have just gone out

    // one phase: quadrant (qa, qb); read half (ro, rh) of stage rs; ask for half (lo, lh) into stage lst
    // (the second operand first in the MFMA: a lane then holds four consecutive columns of one row)
    // (from fragment r0 of that half on; on top the first xn fragments of stage xs's half (0, 1))
#define PM_PHASE(P, qa, qb, rs, ro, rh, r0, xs, xn, lst, lo, lh, cur)                                                \
    do {                                                                                                             \
        constexpr int share_ = S::I(qa), n_ = 4 * share_ * J, half_ = n_ / 2;                                         \
        constexpr int own_ = 4 * ((ro) == 0 ? S::I(rh) : J) - (r0), reads_ = own_ + (xn), loads_ = S::loads(P);       \
        constexpr int rper_ = (reads_ + half_ - 1) / half_, lper_ = (loads_ + half_ - 1) / half_;                     \
        constexpr int lgap_ = half_ / loads_ > 0 ? half_ / loads_ : 1;                                               \
        _Pragma("unroll") for (int s_ = 0; s_ < n_; ++s_) {                                                          \
            const int ks_ = s_ / (share_ * J), i_ = s_ / J % share_, j_ = s_ % J;                                    \
            acc[qa][qb][i_][j_] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[qb][j_][ks_], fa[qa][i_][ks_], acc[qa][qb][i_][j_], 0, 0, 0); \
            __builtin_amdgcn_sched_barrier(0);                                                                       \
            if (s_ < half_) {                                                                                        \
                _Pragma("unroll") for (int x_ = 0; x_ < rper_; ++x_) {                                               \
                    const int r_ = s_ * rper_ + x_;                                                                  \
                    if (r_ < own_) read(rs, ro, rh, (r0) + r_);                                                      \
                    else if (r_ < reads_) read(xs, 0, 1, r_ - own_);                                                 \
                }                                                                                                    \
                __builtin_amdgcn_sched_barrier(0);                                                                   \
            } else if ((s_ - half_) % lgap_ == 0) {                                                                  \
                _Pragma("unroll") for (int x_ = 0; x_ < lper_; ++x_) {                                               \
                    const int l_ = (s_ - half_) / lgap_ * lper_ + x_;                                                \
                    if (l_ < loads_) load(lst, lo, lh, l_, cur);                                                     \
                }                                                                                                    \
                __builtin_amdgcn_sched_barrier(0);                                                                   \
            }                                                                                                        \
        }                                                                                                            \
        /* (until a half that was asked for behind the stores is needed, the stores need not be through) */          \
        if ((P) < 6 && fresh) gemm_phase_wait<S::wait(P) + S::STORES>();                                             \
        else gemm_phase_wait<S::wait(P)>();                                                                          \
        __builtin_amdgcn_sched_barrier(0);                                                                           \
    } while (0)

    int j = blockIdx.x / 8;
    if (!in_range(j)) return;
    // a quarter may lie behind the rows or columns in use (a work-group has one quarter at most): nothing to read or store
    if (p.split == 2) {
        const Where w = locate(j);
        if (w.m0 >= (TA ? p.M : w.rows) || w.n0 >= p.N) return;
    }
    Cursor c0, c1, c2, c3;                        // k-tiles 0 .. 3 from here
    c0.j = j;
    seek(c0);
    c1 = c0; advance(c1);
    c2 = c1; advance(c2);
    c3 = c2; advance(c3);
    auto ask = [&](int stage, int o, int h, const Cursor &c) {
#pragma unroll
        for (int i = 0; i < S::half_loads(o, h); ++i) load(stage, o, h, i, c);
    };
    ask(0, 0, 0, c0);
    ask(0, 1, 0, c0);
    ask(0, 1, 1, c0);
    ask(0, 0, 1, c0);
    ask(1, 0, 0, c1);
    ask(1, 1, 1, c1);
    ask(1, 1, 0, c1);
    ask(1, 0, 1, c1);
    gemm_phase_wait<3 * S::half_loads(1, 0) + 2 * S::half_loads(0, 1) + S::half_loads(0, 0)>();
#pragma unroll
    for (int r = 0; r < 4 * S::I(0); ++r) read(0, 0, 0, r);
#pragma unroll
    for (int r = 0; r < 4 * J; ++r) read(0, 1, 0, r);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    ask(0, 0, 0, c2);
    gemm_phase_wait<S::wait(7)>();
    __builtin_amdgcn_sched_barrier(0);

    Where here = locate(j);
    int left = pairs(k_of(here)), turn = 0;
    // the tile's slice of the bias goes into LDS ahead of the tile's own loads, so it is there with them
    auto ask_bias = [&] {
        if (!GRAD && p.bias && !p.bias_by_value && wave == 0)
            gemm_dma16(gemm_desc(p.bias + (int64_t)here.e * p.N + here.n0, (int64_t)(p.N - here.n0) * 2), lane * 16, 0u, lds0 + S::BIAS + turn * 1024);
    };
    ask_bias();

    auto finish = [&] {                           // the results of the tile to memory
        // (the lane number is hidden from the compiler: what follows from it is worked out here once per tile
        // instead of in registers that the loop over k needs)
        int l = lane;
        asm volatile("" : "+v"(l));
        uint8_t *piece = lds + S::OPERANDS + wave * (32 * S::PITCH);
        const uint8_t *get = piece + l / (4 * J) * S::PITCH + l % (4 * J) * 16;
        uint8_t *lay = piece + (l & 31) * S::PITCH + (l >> 5) * 8;
        // where a lane's 16-byte pieces go, from the tile's corner; the uniform part of a piece's place is the store's scalar offset
        const int put_col = wn * 32 * J + l % (4 * J) * 8;
        const uint32_t put = ((uint32_t)(l / (4 * J)) * (uint32_t)p.ldc + (uint32_t)put_col) * 2u;
        auto row_of = [&](int a, int i) { return S::half(0, 0) * a + 32 * (S::I(a) * wm + i); };      // first row of a wave's fragment in the tile
        const int M = TA ? p.M : here.rows;
        const int64_t corner = (int64_t)here.e * p.sC + (int64_t)here.m0 * p.ldc + here.n0;
        const int bytes = (int)max((int64_t)0, min((int64_t)0x7fffffff, ((int64_t)(M - here.m0 - 1) * p.ldc + (p.N - here.n0)) * 2));
        const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(p.C + corner, 0, bytes, 0x00020000);
        const __amdgpu_buffer_rsrc_t mask = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(GRAD ? p.mask + corner : p.C), 0, GRAD ? bytes : 0, 0x00020000);
        // GRAD: a piece's masks are asked for while the piece before is worked on and ahead of its stores (asked for when
        // they were wanted, each piece waited for memory and for the stores before it: 337 us at 8 x 4096 x 4096 x 1024)
        pm_u32x4 keep[2][2 * J];
        constexpr int PIECES = S::I(0) + S::I(1);
        auto ask = [&](int n) {                   // piece n: half b of the columns, half a of the rows, fragment i
            const int b = n / PIECES, a = n % PIECES >= S::I(0), i = n % PIECES - a * S::I(0);
            const uint32_t at = here.n0 + S::half(1, 0) * b + put_col < p.N ? put : GEMM_NOWHERE;
#pragma unroll
            for (int t = 0; t < 2 * J; ++t)
                keep[n & 1][t] = __builtin_amdgcn_raw_buffer_load_b128(mask, at, ((uint32_t)(row_of(a, i) + 16 / J * t) * (uint32_t)p.ldc + S::half(1, 0) * b) * 2u, 0);
        };
        if (GRAD) ask(0);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const uint32_t put_b = here.n0 + S::half(1, 0) * b + put_col < p.N ? put : GEMM_NOWHERE;
            float add[8];                         // bias of the lane's columns (GRAD: their sums)
#pragma unroll
            for (int x = 0; x < 8; ++x) add[x] = 0.f;
            if (!GRAD && p.bias) {
                if (p.bias_by_value) {
#pragma unroll
                    for (int x = 0; x < 8; ++x) add[x] = bf16_to_f32(p.bias[(int64_t)here.e * p.N + min(here.n0 + S::half(1, 0) * b + put_col + x, p.N - 1)]);
                } else {
                    Elem<PLANMOE_BF16>::unpack(*reinterpret_cast<const uint4 *>(lds + S::BIAS + turn * 1024 + (S::half(1, 0) * b + put_col) * 2), add);
                }
            }
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int i = 0; i < S::I(a); ++i) {
                    auto so = [&](int t) { return ((uint32_t)(row_of(a, i) + 16 / J * t) * (uint32_t)p.ldc + S::half(1, 0) * b) * 2u; };
                    const int n = PIECES * b + S::I(0) * a + i;
                    if (GRAD && n + 1 < 2 * PIECES) ask(n + 1);
#pragma unroll
                    for (int jj = 0; jj < J; ++jj)
                        asm volatile("" : "+a"(acc[a][b][i][jj]));      // (in the accumulator registers until here: copied all at once they would not fit)
#pragma unroll
                    for (int jj = 0; jj < J; ++jj)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const f32x16 &c = acc[a][b][i][jj];
                            *reinterpret_cast<uint2 *>(lay + (32 * jj + 8 * q) * 2) =
                                make_uint2(f32x2_to_bf16x2(c[4 * q], c[4 * q + 1]), f32x2_to_bf16x2(c[4 * q + 2], c[4 * q + 3]));
                        }
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int t = 0; t < 2 * J; ++t) {
                        pm_u32x4 v = *reinterpret_cast<const pm_u32x4 *>(get + t * (16 / J) * S::PITCH);
                        if (!GRAD && p.bias) {    // the matmul's rounding is done; torch.add in bf16
#pragma unroll
                            for (int x = 0; x < 4; ++x)
                                v[x] = f32x2_to_bf16x2(__uint_as_float(v[x] << 16) + add[2 * x], __uint_as_float(v[x] & 0xffff0000u) + add[2 * x + 1]);
                        }
                        if (!GRAD && p.relu) {
#pragma unroll
                            for (int x = 0; x < 4; ++x) v[x] = relu_bf16x2(v[x]);
                        }
                        if (GRAD) {               // relu's backward: kept where its output was positive
#pragma unroll
                            for (int x = 0; x < 4; ++x) {
                                const uint32_t k = keep[n & 1][t][x];
                                v[x] &= ((int)(k << 16) > 0 ? 0xffffu : 0u) | ((int)k >= 0x10000 ? 0xffff0000u : 0u);
                                add[2 * x] += __uint_as_float(v[x] << 16);
                                add[2 * x + 1] += __uint_as_float(v[x] & 0xffff0000u);
                                // (added here: moved to where the sums are wanted, the additions would keep every value of the tile alive)
                                asm volatile("" : "+v"(add[2 * x]), "+v"(add[2 * x + 1]));
                            }
                        }
                        __builtin_amdgcn_raw_buffer_store_b128(v, out, put_b, so(t), 0);
                        // A vector instruction that writes the first register of a 16-byte store right behind it can reach
                        // the stored value (seen with a scalar offset, where the compiler leaves no gap): results of one
                        // column in eight were the next address.  The value is held over a gap.
                        asm volatile("s_nop 1" :: "v"(v));
                        if (GRAD) __builtin_amdgcn_sched_barrier(0);         // (one piece's temporaries at a time: the registers are full)
                    }
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_sched_barrier(0);
                }
            if (GRAD && p.colsum) {
                // the 16 / J lanes that hold a column meet in the wave's piece of LDS
                float *sums = reinterpret_cast<float *>(piece);
                *reinterpret_cast<float4 *>(sums + l * 8) = make_float4(add[0], add[1], add[2], add[3]);
                *reinterpret_cast<float4 *>(sums + l * 8 + 4) = make_float4(add[4], add[5], add[6], add[7]);
                __builtin_amdgcn_wave_barrier();
                float s = 0.f;
                const int c = l % (32 * J);
#pragma unroll
                for (int r = 0; r < 16 / J; ++r) s += sums[(c / 8 + 4 * J * r) * 8 + c % 8];
                const int col = here.n0 + S::half(1, 0) * b + wn * 32 * J + c;
                const int each = S::WM == 2 ? 128 : S::BM, slots = (p.M + each - 1) / each * S::WM, slot = here.m0 / each * S::WM + wm;
                if (l < 32 * J && col < p.N && slot < slots) {
                    float *to = p.colsum + ((int64_t)here.e * slots + slot) * p.N + col;
                    to[0] = s;
                    if (S::WM == 2 && S::BM == 256 && slot + 2 < slots) to[2 * (int64_t)p.N] = 0.f;        // (a tile of 256 rows: all in the first slot)
                }
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    while (true) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int i = 0; i < S::I(a); ++i)
#pragma unroll
                    for (int jj = 0; jj < J; ++jj)
#pragma unroll
                        for (int q = 0; q < 16; ++q) acc[a][b][i][jj][q] = 0.f;
        do {
            PM_PHASE(0, 0, 0, 0, 1, 1, 0, 0, S::EARLY, 0, 1, 0, c2);
            PM_PHASE(1, 0, 1, 0, 0, 1, S::EARLY, 0, 0, 0, 1, 1, c2);
            PM_PHASE(2, 1, 1, 1, 0, 0, 0, 0, 0, 0, 0, 1, c2);
            PM_PHASE(3, 1, 0, 1, 1, 1, 0, 0, 0, 1, 0, 0, c3);
            c2 = c3; advance(c3);
            PM_PHASE(4, 0, 1, 1, 1, 0, 0, 1, S::EARLY, 1, 1, 1, c2);
            PM_PHASE(5, 0, 0, 1, 0, 1, S::EARLY, 0, 0, 1, 1, 0, c2);
            PM_PHASE(6, 1, 0, 0, 0, 0, 0, 0, 0, 1, 0, 1, c2);
            PM_PHASE(7, 1, 1, 0, 1, 0, 0, 0, 0, 0, 0, 0, c3);
            c2 = c3; advance(c3);
            fresh = 0;
        } while (--left);
        finish();
        fresh = 1;
        j += stride;
        if (!in_range(j)) break;
        here = locate(j);
        left = pairs(k_of(here));
        turn ^= 1;
        ask_bias();
    }
    // nothing may still be on its way into LDS that another work-group gets
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#undef PM_PHASE
}

// out[e][c][r] = in[e][r][c] for r < rows, zero for rows <= r < rows_out (the padding of a k dimension):
// 64 x 64 tiles through LDS, 16-byte accesses on both sides
__global__ __launch_bounds__(256) void transpose_bf16_kernel(const uint16_t *__restrict__ in, uint16_t *__restrict__ out,
                                                             int rows, int cols, int rows_out, int64_t s_in, int64_t s_out)
{
    __shared__ uint16_t tile[64][64 + 2];
    const int e = blockIdx.z, r0 = blockIdx.y * 64, c0 = blockIdx.x * 64, tid = threadIdx.x;
    in += (int64_t)e * s_in;
    out += (int64_t)e * s_out;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int q = tid + 256 * i, r = q >> 3, c = (q & 7) * 8;
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (r0 + r < rows && c0 + c < cols) v = *reinterpret_cast<const uint4 *>(in + (int64_t)(r0 + r) * cols + c0 + c);
        uint32_t *dst = reinterpret_cast<uint32_t *>(&tile[r][c]);
        dst[0] = v.x; dst[1] = v.y; dst[2] = v.z; dst[3] = v.w;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int q = tid + 256 * i, c = q >> 3, r = (q & 7) * 8;
        if (c0 + c < cols && r0 + r < rows_out) {
            uint32_t w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = (uint32_t)tile[r + 2 * j][c] | ((uint32_t)tile[r + 2 * j + 1][c] << 16);
            *reinterpret_cast<uint4 *>(out + (int64_t)(c0 + c) * rows_out + r0 + r) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
}

} // namespace pm

using namespace pm;

namespace {

template <class S, bool TA, bool TB, bool GRAD>
int gemm_launch(const GemmArgs &p, hipStream_t stream, const char *who)
{
    const auto kernel = gemm_bf16_kernel<S, TA, TB, GRAD>;
    static bool ready[64];                       // (per device; setting the attribute twice does no harm)
    int dev = 0;
    PM_REQUIRE(hipGetDevice(&dev) == hipSuccess, "%s: no device", who);
    if (dev >= 64 || !ready[dev]) {
        PM_REQUIRE(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS) == hipSuccess,
                   "%s: the kernel needs %d bytes of LDS", who, S::LDS);
        if (dev < 64) ready[dev] = true;
    }
    const int64_t side = p.split == 2 ? 256 : S::BM, side_n = p.split == 2 ? 256 : S::BN;
    int64_t tiles = ((int64_t)p.M + side - 1) / side * (((int64_t)p.N + side_n - 1) / side_n) * p.batches;
    PM_REQUIRE(tiles < ((int64_t)1 << 30), "%s: too many tiles", who);
    if (p.split == 2) tiles = 4 * (tiles < p.stay / 2 ? tiles : p.stay / 2);
    const int64_t stay = (int64_t)compute_units() * S::WAVES_PER_SIMD / 8 * 8;
    kernel<<<dim3((unsigned)(tiles + 7 < stay ? (tiles + 7) / 8 * 8 : stay)), GEMM_WG, S::LDS, stream>>>(p);
    PM_LAUNCH_CHECK(who);
    return 0;
}

// Which tile: 256 x 256 moves the fewest operand bytes per product, 128 x 128 (two work-groups per compute
// unit) leaves fewer compute units idle where there are few tiles and loses less in a last round that is
// not full.  Between them 128, 160 and 192 rows by 256 columns, where the tiles of 256 rows leave compute units idle and 128 x 128
// is bound by its operands: the height whose tiles fill the rounds best.  A launch takes its rounds; a round takes its k-tiles,
// each faster with few compute units at work than with all of them (the clock sinks under the matrix cores), and what a tile
// costs once.  Reading the weights is a floor: what memory gives, or, with few work-groups, what they have on their way (28 GB/s for each
// in 128 x 128, 45 in 256 columns).  Fitted to 450 timings of 110 shapes with the weights in the last cache and out of it: what it picked took
// 1.1 % longer than the best, before there was a tile of 128 x 64 (gemm_pick takes 0.72 of small() for it, the weight's floor in it included, which
// is what half the columns on twice the compute units give in gemm_is_deep's table).
// us in one launch, rows +- sqrt(rows) in use, nn:
//   experts x rows, in, out      128 x 128    256    128    160    192 x 256
//   8 x 500, 2048, 2048             49         48     57     42     42     (54 in 256 and a launch of quarters)
//   8 x 128, 4096, 4096             84         80     64     64     66
//   16 x 512, 1024, 1024            29         31     34     25     26
//   8 x 250, 2048, 2048             31         43     29     32     35
//   8 x 2000, 4096, 1024           142        171    158    129    140
//   8 x 4096, 4096, 4096          1125        846    987    968    930
//   8 x 110, 2688, 2560             36         58     52     54     55     (weights cold)
//   8 x 60, 1024, 4096              19         29     23     25     26     (weights cold)
//
// A last round of large tiles that is at most half full may be a launch of its own, in quarters (8 experts of 4096 +- 100
// rows by 1024 columns: 512 tiles and a few, whose third round would take half as long again as the other two).
struct GemmCost {
    double rows, kt, cu;                         // rows expected of a batch; k-tiles
    int64_t most, n, batches, weight_bytes;      // rows at most
    bool counted;                                // the rows are an expectation: of many batches, with a standard deviation of its root

    double tiles(int64_t bm, int64_t bn) const
    {
        double t = 0;
        for (const double q : {-1.5, -0.5, 0.5, 1.5}) {
            const int64_t r = counted ? std::min(most, std::max<int64_t>(1, (int64_t)(rows + q * std::sqrt(rows)))) : (int64_t)rows;
            t += 0.25 * (double)((r + bm - 1) / bm);
        }
        return t * (double)((n + bn - 1) / bn * batches);
    }
    double rounds(double t, double low, double high, double once) const
    {
        const double full = std::floor(t / cu), rest = t - full * cu;
        return full * (high * kt + once) + (rest > 0.01 ? (low + (high - low) * rest / cu) * kt + once : 0.);
    }
    double quarters(double t) const              // tiles of 128 x 128, two work-groups per compute unit
    {
        const double full = std::floor(t / (2 * cu)), rest = t - full * 2 * cu;
        return full * (kt + 2) + (rest <= 0.01 ? 0. : rest <= cu ? (0.41 + 0.19 * rest / cu) * kt + 2 : (0.85 + 0.25 * (rest - cu) / cu) * kt + 2);
    }
    // reading the weights: what memory gives, or what the tiles' columns that are worked on ask for, each `each` TB/s
    double floor(double t, int bn, double each, double once) const
    {
        const double columns = (double)((n + bn - 1) / bn * batches) * std::min(1., cu / t);
        return (double)weight_bytes * 1e-6 / std::min(4.8, each * columns) + once;
    }
    double small() const
    {
        const double t = tiles(128, 128);
        return std::max(quarters(t) + 4.5, t <= cu ? floor(t, 128, 0.028, 5.5) : (double)weight_bytes * 1e-6 / 3.5 + 6);
    }
    double big() const
    {
        const double t = tiles(256, 256);
        return std::max(rounds(t, 1.0, 1.4, 3) + 6, floor(t, 256, 0.045, 8));
    }
    // the last round as a launch of quarters; with many rounds it hardly counts
    double big_and_quarters() const
    {
        const double t = tiles(256, 256), full = std::floor(t / cu), last = t - full * cu;
        return t < 6 * cu && full > 0 && last > 0.01 && 2 * last <= cu ? std::max(full * (1.4 * kt + 3) + 6 + quarters(4 * last) + 10, floor(t, 256, 0.045, 8)) : 1e30;
    }
    double low(int height) const                 // height: 128, 160, 192
    {
        const double t = tiles(height, 256), us = height == 128 ? rounds(t, 0.58, 0.9, 2) : height == 160 ? rounds(t, 0.7, 1.07, 2) : rounds(t, 0.79, 1.25, 2);
        return std::max(us + 6, floor(t, 256, 0.045, 6));
    }
};

// The column sums of a masked product: a tile of so many rows has so many slots (0 rows: one slot for everything)
struct GemmSlots { int rows, per_tile; };

// Few rows per batch against a whole weight.  Up to 16 rows always, and up to 32 where there is a compute unit for each
// work-group: beyond that a tile's operands, read once for all its rows, win.
// us, cold weights, few rows and tiles, nn, nt:
//   8 x 40 rows, 2688 -> 2560     35, 33 and 30, 27      8 x 20, same       29, 28 and 32, 28
//   16 x 40, 2688 -> 2560         66, 62 and 53, 47      16 x 20, same      56, 52 and 52, 46
//   16 x 40, 1024 -> 4096         37, 36 and 31, 29      8 x 20, same       17, 16 and 19, 17
//   8 x 40, 4096 -> 1024          35, 32 and 36, 34      8 x 8 2688 -> 2560 26, 25 and 32, 28
bool gemm_is_skinny(bool nt, int m, int n, int64_t k, int batches)
{
    if (m > SKINNY_ROWS || batches > 65535 || n * k * 2 >= ((int64_t)1 << 31)) return false;
    const int width = gemm_skinny_width(nt, n, k, batches);
    return m <= 16 || (int64_t)((n + width - 1) / width) * batches <= compute_units();
}

// 128 x 128 with a compute unit for each tile (gemm_deep.hip).  Not up to the last one: with rows up to the capacity a few experts have a
// tile more than expected, and two of these work-groups do not fit on a compute unit.  us in gemm_bf16_kernel's 128 x 128 tiles and here, weights cold, in cache:
//   8 experts x 80 rows, 4096 -> 1024    43, 33 and 41, 25      8 x 80, 1024 -> 512     13, 13 and 9, 9
//   8 x 110, 2696 -> 2488                39, 32 and 37, 29      a^T b, 4 x 512 x 768 over 2000 rows    20 and 15
// In 64 columns where that leaves a compute unit for each tile still: half of the weight for each, and five k-tiles on their way instead of four.
// us in 128 and 64 columns, weights cold, nn and nt:
//   8 x 32 rows, 4096 -> 1024            35.6, 26.8 and 34.3, 24.1      8 x 128, same            42.1, 34.9 and 39.5, 29.4
//   8 x 32, 2048 -> 2048                 23.7, 17.6 and 21.5, 18.1      16 x 64, 1024 -> 1024    14.0, 11.6 and 13.1, 10.1
//   4 x 64, 512 -> 2048                  8.8, 7.1 and 8.6, 6.6          4 x 256, 2048 -> 512     22.9, 18.0 and 21.2, 15.6
//   4 x 64, 4096 -> 4096                 40.0, 32.6 and 41.6, 32.6      a^T b, 4 x 512 x 768 over 256 rows    6.7, 5.4
// (four k-tiles: 8 x 32, 4096 -> 1024 30.9 and 29.7; six: the same as five there, 4 x 64, 4096 -> 4096 37.3)
bool gemm_is_deep(double tiles, int m) { return tiles <= 0.8 * compute_units() || (m <= 128 && tiles <= compute_units()); }

enum GemmKernel { GEMM_SKINNY, GEMM_DEEP, GEMM_DEEP_64, GEMM_128, GEMM_LOW_128, GEMM_LOW_160, GEMM_LOW_192, GEMM_256, GEMM_256_QUARTERS };

// form: 0 nn, 1 nt, 2 tn; contiguous: the operands and the result are; rows: expected of a batch (tn: of its reduction)
GemmKernel gemm_pick(int form, bool contiguous, int m, int n, int k, int batches, bool counted, int64_t rows)
{
    const bool tn = form == 2;
    if (!tn && contiguous && gemm_is_skinny(form == 1, m, n, k, batches)) return GEMM_SKINNY;
    const GemmCost cost{(double)(tn ? m : rows), (double)(((tn ? rows : k) + 63) / 64), (double)compute_units(), m, n, batches,
                        tn ? 0 : (int64_t)n * k * batches * 2, !tn && counted};
    const bool deep = contiguous && gemm_is_deep(cost.tiles(128, 128), m) && gemm_deep_reaches(form, m, n, k);
    const bool narrow = deep && gemm_is_deep(cost.tiles(128, 64), m);
    const double small = (narrow ? 0.72 : deep ? 0.88 : 1.) * cost.small(), split = cost.big_and_quarters(), big = std::min(cost.big(), split);
    if (!tn) {
        const double low[3] = {cost.low(128), cost.low(160), cost.low(192)};
        const int f = low[0] <= low[1] && low[0] <= low[2] ? 0 : low[1] <= low[2] ? 1 : 2;
        if (low[f] < small && low[f] < big) return f == 0 ? GEMM_LOW_128 : f == 1 ? GEMM_LOW_160 : GEMM_LOW_192;
    }
    if (small < big) return narrow ? GEMM_DEEP_64 : deep ? GEMM_DEEP : GEMM_128;
    return big == split ? GEMM_256_QUARTERS : GEMM_256;
}

bool gemm_contiguous(int form, int m, int n, int k, int lda, int ldb, int ldc, int64_t sa, int64_t sb, int64_t sc)
{
    return lda == (form == 2 ? m : k) && ldb == (form == 1 ? k : n) && ldc == n && sb == (int64_t)n * k && sa == (int64_t)m * k && sc == (int64_t)m * n;
}

GemmSlots gemm_slots(GemmKernel kernel)
{
    switch (kernel) {
    case GEMM_SKINNY: return GemmSlots{0, 1};
    case GEMM_LOW_128: return GemmSlots{128, 1};
    case GEMM_LOW_160: return GemmSlots{160, 1};
    case GEMM_LOW_192: return GemmSlots{192, 1};
    default: return GemmSlots{128, 2};
    }
}

template <bool TA, bool TB, bool GRAD>
int gemm_run(GemmArgs p, int64_t rows_hint, hipStream_t stream, const char *who, GemmSlots *sums = nullptr)
{
    constexpr int form = TA ? 2 : TB ? 0 : 1;
    const bool contiguous = gemm_contiguous(form, p.M, p.N, p.K, p.lda, p.ldb, p.ldc, p.sA, p.sB, p.sC);
    const SkinnyArgs few{p.A, p.B, p.bias, p.mask, p.C, p.colsum, p.live, p.live_planes, p.live_round, p.M, p.N, p.K, p.batches, p.relu};
    const GemmKernel kernel = gemm_pick(form, contiguous, p.M, p.N, p.K, p.batches, p.live, rows_hint);
    if (sums) *sums = gemm_slots(kernel);
    if constexpr (!TA) {
        if (kernel == GEMM_SKINNY) return gemm_skinny_run(!TB, few, stream, who);
        if (kernel == GEMM_LOW_128) return gemm_launch<GemmFlat<2, 2>, TA, TB, GRAD>(p, stream, who);
        if (kernel == GEMM_LOW_160) return gemm_launch<GemmFlat<2, 3>, TA, TB, GRAD>(p, stream, who);
        if (kernel == GEMM_LOW_192) return gemm_launch<GemmFlat<3, 3>, TA, TB, GRAD>(p, stream, who);
    }
    if (kernel == GEMM_DEEP || kernel == GEMM_DEEP_64) return gemm_deep_run(form, kernel == GEMM_DEEP ? 128 : 64, few, stream, who);
    if (kernel == GEMM_128) return gemm_launch<Gemm128, TA, TB, GRAD>(p, stream, who);
    p.stay = compute_units() / 8 * 8;
    p.split = kernel == GEMM_256_QUARTERS;
    if (gemm_launch<Gemm256, TA, TB, GRAD>(p, stream, who)) return 1;
    if (!p.split) return 0;
    p.split = 2;
    return gemm_launch<Gemm128, TA, TB, GRAD>(p, stream, who);
}

}  // namespace

// In shares (layer_shares.hip): where the work-groups that the weight's columns make, for the experts that can have rows, leave half of the compute
// units without one.  Up to 32 rows 64 columns (whole lines of 128 bytes) and shares of at least 512 k, 16 steps for 16 waves; beyond, tiles of
// 128 x 128 and shares of at least 4 k-tiles.  Up to eight: the combine reads them all.
GemmShares pm::gemm_shares_pick(int m, int n, int64_t k, int batches, int64_t rows, int64_t pairs, int64_t most)
{
    const int64_t cu = compute_units();
    const int active = (int)std::min<int64_t>(batches, pairs);
    if (n * k * 2 >= ((int64_t)1 << 31) || batches > 64) return GemmShares{};
    if (gemm_is_skinny(false, m, n, k, batches)) {
        const int64_t groups = (int64_t)((n + 63) / 64) * active, splits = std::min<int64_t>({groups > 0 ? cu / groups : 0, k / 512, 8, most});
        // (one share: where fewer experts than there are have rows, and the whole product would take them in wider columns)
        if (splits >= 2 || (splits == 1 && active < batches && gemm_skinny_width(false, n, k, batches) > 64)) return GemmShares{(int)splits, active, true};
        return GemmShares{};
    }
    if (!gemm_deep_reaches(0, m, n, k)) return GemmShares{};
    const double tiles = GemmCost{(double)std::min<int64_t>(rows, m), 0., (double)cu, m, n, batches, 0, true}.tiles(128, 128);
    const int64_t k_tiles = (k + DEEP_BK - 1) / DEEP_BK, splits = std::min<int64_t>({(int64_t)((double)cu / tiles), k_tiles / 4, 8, most});
    if (splits < 2) return GemmShares{};
    const int64_t each = (k_tiles + splits - 1) / splits;
    return GemmShares{(int)((k_tiles + each - 1) / each), active, false};      // (none of them empty)
}

// Product and combine together, against the whole product (in 32 or 64 columns, where that leaves compute units without a tile) and the
// combine of its rows.  Up to 32 rows: from 1536 k on; from 1024 on where fewer experts than there are have rows.  Tiles: the k-tiles that a
// work-group has fewer, 0.2 us each, against 2 us and 0.3 for every MB of shares; with no more work-groups than the whole product has of tiles of 64
// columns only where an expert's rows are a whole tile's and more (its weight is read by half as many).  Through the codec a wave adds up a row's
// shares, 512 values at a time: 1.5 us each, twice that with more than four; for few rows, whose whole product takes less, only rows of up to
// 512, or 1024 with a reduction of 4096.  Top-2, us whole and in shares, weights in the last cache and cold, without the codec, then through it:
//   8 experts, 4096 -> 1024     4 tokens 14.4, 14.7 and 22.3, 16.2     128: 21.2, 18.9 and 31.3, 22.5     512: 26.6, 23.7 and 40.5, 32.2
//                                        15.4, 17.8     23.1, 19.3          22.0, 22.1     32.1, 25.8          27.6, 26.8     41.0, 35.2
//   4 experts, 2048 -> 512      4        9.7, 7.7       10.1, 8.1      128: 13.1, 12.7     14.4, 12.9     512: 13.9, 17.5     16.5, 17.7 *
//                                        9.9, 8.6       10.4, 9.0           13.4, 13.6     14.7, 13.8 *        14.2, 18.3     16.7, 18.5 *
//   8 experts, 2048 -> 2048     1        9.7, 7.8       13.9, 9.9      128: 17.6, 18.5     22.3, 23.0 *   400: 21.0, 21.7     25.9, 25.6
//                                        11.2, 13.5     15.5, 15.8 *        19.2, 26.8     23.8, 31.4 *        22.7, 29.3     27.4, 33.3 *
//   4 experts, 1024 -> 1024     1        7.1, 7.1       7.2, 7.4       128: 10.7, 11.6     11.4, 11.8 *   512: 11.9, 19.1     12.8, 18.9 *
//   16 experts, 4096 -> 1024    256      27.8, 28.5     34.8, 37.2 *   (* computed whole)
// 254 shapes (256 to 4096 columns, 512 to 4096 k, 1 to 2048 tokens), against the whole product each: 0.91 in the last cache, 0.81 cold; with the shares wherever
// they fit 0.95 and 0.82, through the codec 1.14 and 0.97, now 0.96 and 0.89.
bool pm::gemm_shares_pay(const GemmShares &how, int m, int n, int64_t k, int batches, int64_t rows, int64_t pairs, bool coded)
{
    if (how.splits == 0) return false;
    if (how.few) {
        if (coded && !(n <= 512 || (n <= 1024 && k >= 4096))) return false;
        return k >= 1536 || (k >= 1024 && how.active < batches);
    }
    const GemmCost cost{(double)std::min<int64_t>(rows, m), 0., (double)compute_units(), m, n, batches, 0, true};
    const int64_t k_tiles = (k + DEEP_BK - 1) / DEEP_BK, each = (k_tiles + how.splits - 1) / how.splits;
    if (how.splits * cost.tiles(128, 128) < 1.25 * cost.tiles(128, 64)) return rows > 96 && (coded ? k_tiles >= 64 && n <= 1024 : k_tiles >= 32);
    const double mb = 4e-6 * how.splits * n * (double)std::min<int64_t>(pairs, (int64_t)batches * m);
    return 0.2 * (double)(k_tiles - each) > 2. + 0.3 * mb + (coded ? 1.5 * ((n + 511) / 512) * (how.splits > 4 ? 2 : 1) : 0.);
}

int pm::gemm_shares_run(const GemmShares &how, SkinnyArgs p, hipStream_t stream, const char *who)
{
    p.splits = how.splits;
    p.active = how.active;
    return how.few ? gemm_skinny_shares_run(p, stream, who) : gemm_deep_shares_run(p, stream, who);
}

namespace {

// what the buffer descriptors cover: from a tile's corner, a tile of a k-fast operand and 64 rows of a k-slow one
bool gemm_pitch_fits(int ld) { return (int64_t)ld * 2 * 256 < ((int64_t)1 << 31); }

}  // namespace

extern "C" int planmoe_gemm_nt_bf16(const void *a, const void *b, const void *bias, int activation, int batches,
                                    int m, int n, int k, int lda, int ldb, int ldc, int64_t batch_stride_a,
                                    int64_t batch_stride_b, int64_t batch_stride_c, void *c, void *stream)
{
    PM_REQUIRE(batches >= 0 && m >= 0 && n >= 0 && k >= 1, "planmoe_gemm_nt_bf16: bad shape");
    if (batches == 0 || m == 0 || n == 0) return 0;
    PM_REQUIRE(a && b && c, "planmoe_gemm_nt_bf16: NULL argument");
    PM_REQUIRE(activation == 0 || activation == 1, "planmoe_gemm_nt_bf16: activation is 0 (none) or 1 (relu)");
    PM_REQUIRE(k % 8 == 0 && n % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0 && ldc % 8 == 0 && lda >= k && ldb >= k && ldc >= n,
               "planmoe_gemm_nt_bf16: k, n and the row pitches must be multiples of 8 (16-byte pieces); pitches cover their rows");
    PM_REQUIRE(batch_stride_a % 8 == 0 && batch_stride_b % 8 == 0 && batch_stride_c % 8 == 0 && aligned16(a) && aligned16(b) && aligned16(c),
               "planmoe_gemm_nt_bf16: operands must be 16-byte aligned");
    PM_REQUIRE(gemm_pitch_fits(lda) && gemm_pitch_fits(ldb) && gemm_pitch_fits(ldc), "planmoe_gemm_nt_bf16: 256 rows of an operand must stay under 2 GiB");
    GemmArgs p{(const uint16_t *)a, (const uint16_t *)b, (const uint16_t *)bias, nullptr, (uint16_t *)c, nullptr, nullptr, 0, 1, m, n, k,
               lda, ldb, ldc, batch_stride_a, batch_stride_b, batch_stride_c, batches, activation, 0, 0, !aligned16(bias)};
    return gemm_run<false, false, false>(p, m, (hipStream_t)stream, "planmoe_gemm_nt_bf16");
}

extern "C" int planmoe_gemm_nn_bf16(const void *a, const void *b, const void *bias, int activation, int batches,
                                    int m, int n, int k, int lda, int ldb, int ldc, int64_t batch_stride_a,
                                    int64_t batch_stride_b, int64_t batch_stride_c, void *c, void *stream)
{
    PM_REQUIRE(batches >= 0 && m >= 0 && n >= 0 && k >= 64, "planmoe_gemm_nn_bf16: bad shape");
    if (batches == 0 || m == 0 || n == 0) return 0;
    PM_REQUIRE(a && b && c, "planmoe_gemm_nn_bf16: NULL argument");
    PM_REQUIRE(activation == 0 || activation == 1, "planmoe_gemm_nn_bf16: activation is 0 (none) or 1 (relu)");
    PM_REQUIRE(k % GEMM_BK == 0, "planmoe_gemm_nn_bf16: k must be a multiple of %d", GEMM_BK);
    PM_REQUIRE(n % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0 && ldc % 8 == 0 && lda >= k && ldb >= n && ldc >= n,
               "planmoe_gemm_nn_bf16: n and the row pitches must be multiples of 8 (16-byte pieces); pitches cover their rows");
    PM_REQUIRE(batch_stride_a % 8 == 0 && batch_stride_b % 8 == 0 && batch_stride_c % 8 == 0 && aligned16(a) && aligned16(b) && aligned16(c),
               "planmoe_gemm_nn_bf16: operands must be 16-byte aligned");
    PM_REQUIRE(gemm_pitch_fits(lda) && gemm_pitch_fits(ldb) && gemm_pitch_fits(ldc), "planmoe_gemm_nn_bf16: 256 rows of an operand must stay under 2 GiB");
    GemmArgs p{(const uint16_t *)a, (const uint16_t *)b, (const uint16_t *)bias, nullptr, (uint16_t *)c, nullptr, nullptr, 0, 1, m, n, k,
               lda, ldb, ldc, batch_stride_a, batch_stride_b, batch_stride_c, batches, activation, 0, 0, !aligned16(bias)};
    return gemm_run<false, true, false>(p, m, (hipStream_t)stream, "planmoe_gemm_nn_bf16");
}

extern "C" int planmoe_gemm_tn_bf16(const void *a, const void *b, int batches, int m, int n, int k, int lda, int ldb,
                                    int ldc, int64_t batch_stride_a, int64_t batch_stride_b, int64_t batch_stride_c,
                                    void *c, void *stream)
{
    PM_REQUIRE(batches >= 0 && m >= 0 && n >= 0 && k >= 64, "planmoe_gemm_tn_bf16: bad shape");
    if (batches == 0 || m == 0 || n == 0) return 0;
    PM_REQUIRE(a && b && c, "planmoe_gemm_tn_bf16: NULL argument");
    PM_REQUIRE(k % GEMM_BK == 0, "planmoe_gemm_tn_bf16: k must be a multiple of %d", GEMM_BK);
    PM_REQUIRE(m % 8 == 0 && n % 8 == 0 && lda % 8 == 0 && ldb % 8 == 0 && ldc % 8 == 0 && lda >= m && ldb >= n && ldc >= n,
               "planmoe_gemm_tn_bf16: m, n and the row pitches must be multiples of 8 (16-byte pieces); pitches cover their rows");
    PM_REQUIRE(batch_stride_a % 8 == 0 && batch_stride_b % 8 == 0 && batch_stride_c % 8 == 0 && aligned16(a) && aligned16(b) && aligned16(c),
               "planmoe_gemm_tn_bf16: operands must be 16-byte aligned");
    PM_REQUIRE(gemm_pitch_fits(lda) && gemm_pitch_fits(ldb) && gemm_pitch_fits(ldc), "planmoe_gemm_tn_bf16: 256 rows of an operand must stay under 2 GiB");
    GemmArgs p{(const uint16_t *)a, (const uint16_t *)b, nullptr, nullptr, (uint16_t *)c, nullptr, nullptr, 0, 1, m, n, k,
               lda, ldb, ldc, batch_stride_a, batch_stride_b, batch_stride_c, batches, 0, 0, 0, false};
    return gemm_run<true, true, false>(p, k, (hipStream_t)stream, "planmoe_gemm_tn_bf16");
}

// ---------------------------------------------------------------- the experts' products on contiguous buffers
int pm::expert_gemm_check(const char *who, int form, int dtype, const void *a, const void *b, int batches, int m, int n, int k,
                          const int32_t *live, int live_planes, int live_round, const void *c)
{
    PM_REQUIRE(form >= 0 && form <= 2, "%s: form is 0 (a b), 1 (a b^T) or 2 (a^T b)", who);
    PM_REQUIRE(dtype == PLANMOE_BF16 || dtype == PLANMOE_F32, "%s: bf16 or fp32", who);
    PM_REQUIRE(batches >= 1 && m >= 1 && n >= 1 && k >= 1, "%s: bad shape", who);
    PM_REQUIRE(a && b && c && aligned16(a) && aligned16(b) && aligned16(c), "%s: NULL or unaligned operand", who);
    const int vec = dtype == PLANMOE_F32 ? 4 : 8;
    // (what is read and stored in 16-byte pieces: the fast index of every operand and of the result)
    PM_REQUIRE(n % vec == 0 && (form == 2 ? m : k) % vec == 0, "%s: the fast index of every operand must be a multiple of %d", who, vec);
    PM_REQUIRE(!live || (batches <= 64 && live_planes >= 1 && live_round >= 1), "%s: row counts for up to 64 batches", who);
    // row lengths: a's, and the longer of b's and c's (n, or with b^T: k and n).  How many rows there are is no row length: the
    // kernels' offsets start at a tile's corner
    const int pitch_a = form == 2 ? m : k, pitch = n > pitch_a ? n : pitch_a;
    PM_REQUIRE((int64_t)pitch * 2 * 256 * (dtype == PLANMOE_F32 ? 2 : 1) < ((int64_t)1 << 31), "%s: 256 rows of an operand must stay under 2 GiB", who);
    return 0;
}

extern "C" int planmoe_expert_gemm(int form, int dtype, const void *a, const void *b, const void *bias, int activation,
                                   int batches, int m, int n, int k, const int32_t *live, int live_planes, int live_round,
                                   int rows_hint, void *c, void *stream)
{
    const char *who = "planmoe_expert_gemm";
    if (expert_gemm_check(who, form, dtype, a, b, batches, m, n, k, live, live_planes, live_round, c)) return 1;
    PM_REQUIRE(activation == 0 || activation == 1, "%s: activation is 0 (none) or 1 (relu)", who);
    PM_REQUIRE(!bias || form != 2, "%s: a weight gradient has no bias", who);
    hipStream_t st = (hipStream_t)stream;
    const int most = form == 2 ? k : m, hint = rows_hint >= 1 && rows_hint < most ? rows_hint : most;
    const OuterArgs outer{a, b, c, live, live_planes, live_round, m, n, k, batches};
    if (dtype == PLANMOE_F32) {
        Gemm32Args p{(const float *)a, (const float *)b, (const float *)bias, nullptr, (float *)c, nullptr, live, live_planes, live_round,
                     m, n, k, batches, activation};
        const Gemm32Kernel kernel = gemm_f32_pick(form, p, hint);
        // (products in parts only: the fp32 tiles have other sums)
        if (form == 2 && kernel >= G32_SPLIT_64 && gemm_outer_serves(dtype, m, n, k, batches, hint)) return gemm_outer_run(dtype, outer, st, who);
        return gemm_f32_run(form, p, kernel, hint, st, who);
    }
    if (form == 2 && !activation && gemm_outer_serves(dtype, m, n, k, batches, hint)) return gemm_outer_run(dtype, outer, st, who);
    const int lda = form == 2 ? m : k, ldb = form == 1 ? k : n;
    GemmArgs p{(const uint16_t *)a, (const uint16_t *)b, (const uint16_t *)bias, nullptr, (uint16_t *)c, nullptr, live, live_planes,
               live_round, m, n, k, lda, ldb, n, (int64_t)m * k, (int64_t)n * k, (int64_t)m * n, batches, activation, 0, 0, !aligned16(bias)};
    if (form == 0) return gemm_run<false, true, false>(p, hint, st, who);
    if (form == 1) return gemm_run<false, false, false>(p, hint, st, who);
    return gemm_run<true, true, false>(p, hint, st, who);
}

extern "C" const char *planmoe_expert_gemm_kernel(int form, int dtype, int activation, int batches, int m, int n, int k, int counted, int rows_hint)
{
    const char *who = "planmoe_expert_gemm_kernel";
    static const int32_t __attribute__((aligned(16))) some[1] = {0};         // (stands for the operands, which are not read)
    const int32_t *live = counted ? some : nullptr;
    auto bad = [&]() -> int {
        if (expert_gemm_check(who, form, dtype, some, some, batches, m, n, k, live, 1, 1, some)) return 1;
        PM_REQUIRE(activation == 0 || activation == 1, "%s: activation is 0 (none) or 1 (relu)", who);
        return 0;
    };
    if (bad()) return nullptr;
    const int most = form == 2 ? k : m, hint = rows_hint >= 1 && rows_hint < most ? rows_hint : most;
    if (dtype == PLANMOE_F32) {
        static const char *const names[] = {"f32 waves", "f32 64x64", "f32 64x64 four stages", "f32 32x32", "f32 32x32 eight stages", "f32 128x128", "f32 parts 64x64", "f32 parts 128x128", "f32 parts 256x128"};
        const Gemm32Kernel kernel = gemm_f32_pick(form, Gemm32Args{nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, live, 1, 1, m, n, k, batches, activation}, hint);
        return form == 2 && kernel >= G32_SPLIT_64 && gemm_outer_serves(dtype, m, n, k, batches, hint) ? "f32 parts few rows of a^T b" : names[kernel];
    }
    if (form == 2 && !activation && gemm_outer_serves(dtype, m, n, k, batches, hint)) return "few rows of a^T b";
    static const char *const names[] = {"few rows", "128x128 alone", "128x128 alone", "128x128", "128x256", "160x256", "192x256", "256x256", "256x256 and quarters"};
    const int lda = form == 2 ? m : k, ldb = form == 1 ? k : n;
    return names[gemm_pick(form, gemm_contiguous(form, m, n, k, lda, ldb, n, (int64_t)m * k, (int64_t)n * k, (int64_t)m * n), m, n, k, batches, counted, hint)];
}

extern "C" size_t planmoe_expert_gemm_relu_bwd_workspace_bytes(int batches, int m, int n)
{
    if (batches < 1 || m < 1 || n < 1) return 16;
    return (size_t)batches * 2 * ((m + 63) / 64) * n * 4;      // (fp32 tiles may have 64 rows)
}

int pm::relu_bwd_with(const char *who, int dtype, const void *a, const void *b, const void *h, int batches, int m, int n, int k, const int *live,
                      int live_planes, int live_round, int rows_hint, void *c, void *dbias, void *workspace, size_t workspace_bytes,
                      const SumJob *others, int others_n, hipStream_t st)
{
    if (expert_gemm_check(who, 1, dtype, a, b, batches, m, n, k, live, live_planes, live_round, c)) return 1;
    PM_REQUIRE(h && aligned16(h), "%s: NULL or unaligned activations", who);
    PM_REQUIRE(!dbias || (workspace && aligned16(workspace) && workspace_bytes >= planmoe_expert_gemm_relu_bwd_workspace_bytes(batches, m, n)), "%s: workspace too small", who);
    PM_REQUIRE(batches <= 65535, "%s: too many batches", who);
    float *parts = dbias ? (float *)workspace : nullptr;
    const int hint = rows_hint >= 1 && rows_hint < m ? rows_hint : m;
    GemmSlots sums;
    if (dtype == PLANMOE_F32) {
        Gemm32Args p{(const float *)a, (const float *)b, nullptr, (const float *)h, (float *)c, parts, live, live_planes, live_round, m, n, k, batches, 0};
        const Gemm32Kernel kernel = gemm_f32_pick(1, p, hint);
        sums = GemmSlots{gemm_f32_slot_rows(kernel), 2};
        if (gemm_f32_run(1, p, kernel, hint, st, who)) return 1;
    } else {
        GemmArgs p{(const uint16_t *)a, (const uint16_t *)b, nullptr, (const uint16_t *)h, (uint16_t *)c, parts, live, live_planes, live_round,
                   m, n, k, k, k, n, (int64_t)m * k, (int64_t)n * k, (int64_t)m * n, batches, 0, 0, 0, false};
        if (gemm_run<false, false, true>(p, hint, st, who, &sums)) return 1;
    }
    SumJob jobs[SUM_JOBS];
    int count = 0;
    for (int i = 0; i < others_n; ++i) jobs[count++] = others[i];
    if (dbias) {
        if (sums.rows == 0) sums.rows = m;
        const int slots = (m + sums.rows - 1) / sums.rows * sums.per_tile;
        jobs[count++] = SumJob{parts, dbias, batches, slots, n, live, live_planes, live_round, m, sums.rows, sums.per_tile};
    }
    return sum_slots(who, dtype, jobs, count, st);
}

extern "C" int planmoe_expert_gemm_relu_bwd(int dtype, const void *a, const void *b, const void *h, int batches, int m, int n,
                                            int k, const int32_t *live, int live_planes, int live_round, int rows_hint, void *c,
                                            void *dbias, void *workspace, size_t workspace_bytes, void *stream)
{
    return relu_bwd_with("planmoe_expert_gemm_relu_bwd", dtype, a, b, h, batches, m, n, k, live, live_planes, live_round, rows_hint, c, dbias, workspace,
                         workspace_bytes, nullptr, 0, (hipStream_t)stream);
}

extern "C" int planmoe_transpose_bf16(const void *in, int batches, int rows, int cols, int rows_out, void *out, void *stream)
{
    PM_REQUIRE(batches >= 0 && rows >= 0 && cols >= 0 && rows_out >= rows, "planmoe_transpose_bf16: bad shape");
    if (batches == 0 || cols == 0 || rows_out == 0) return 0;
    PM_REQUIRE(in && out, "planmoe_transpose_bf16: NULL argument");
    PM_REQUIRE(cols % 8 == 0 && rows_out % 8 == 0 && aligned16(in) && aligned16(out),
               "planmoe_transpose_bf16: cols and rows_out must be multiples of 8, buffers 16-byte aligned");
    PM_REQUIRE((rows_out + 63) / 64 <= 65535 && batches <= 65535, "planmoe_transpose_bf16: too many tiles");
    const dim3 grid((unsigned)((cols + 63) / 64), (unsigned)((rows_out + 63) / 64), (unsigned)batches);
    transpose_bf16_kernel<<<grid, 256, 0, (hipStream_t)stream>>>((const uint16_t *)in, (uint16_t *)out, rows, cols, rows_out,
                                                                 (int64_t)rows * cols, (int64_t)cols * rows_out);
    PM_LAUNCH_CHECK("planmoe_transpose_bf16");
    return 0;
}
