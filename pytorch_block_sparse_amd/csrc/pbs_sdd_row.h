// dense^T x dense -> block-sparse (weight gradient on the sparse support), and with it the bias gradient:
//   out[32b + j][i] = sum_t G[t][32r + i] * X[t][32c + j]   for every data block b at (r, c),   bias[n] = sum_t G[t][n].
//
// A workgroup takes a unit, up to six blocks of one block row of W, over one slice of the tokens (in fp32, where the slices do not
// fit the workspace, of a launch's range of them: a later launch adds to what it finds); each of its four waves
// every fourth chunk of 32 tokens, with all accumulators of the unit (16 registers a block), so that nothing is shared until the
// waves' sums meet in LDS at the end: no barrier and no wait for another wave in the loop, any shape of pattern makes
// units of one size, and small problems have many workgroups.  A G fragment is read once for all products of a unit.
//
// What bounds it: the texture path that copies memory to LDS (a KB costs it 23 cycles in 128-byte rows, 35 in 64-byte ones)
// and the matrix pipe.  fp32: 256 cycles of products per block and chunk against 4 + 4 / NB copies of 23 each: near the matrix rate
// if copies and products overlap, so every copy is issued between two products (issued in a burst, all waves of a CU
// copy together, then compute together: twice the time).  A piece of LDS (32 tokens x 32 features) is refilled as soon as
// its fragments are in registers, and the registers as soon as their product is issued: five pieces per wave hold one
// to four blocks of copies in flight.  bf16: 32 cycles of products against 2 x 35 of copies: bound by the copies, still
// better than rectangles until the operands outgrow the L2s.
// Fragments: fp32 as float2 of two features (the two 16-feature halves of a product are the even and the odd features: one
// 8-byte read serves both); bf16 through transposing reads, the halves chosen so that eight result columns meet in a lane.
//
// Measured, us, against the kernels it replaced (fp32: equal shares of bands of 16 rows, barriers; bf16: rectangles):
//   fp32 768 -> 3072 density 0.5, 4096 tokens 123 -> 96, 1024 tokens 56 -> 30;  3072 -> 768 density 0.25 with uneven rows, 4096 tokens
//   78 -> 50;  768 -> 768 density 0.5, 16384 tokens 122 -> 98;  4096 -> 4096 density 0.25, 16384 tokens 1250 -> 1129 (122 of
//   155 TFLOP/s);  3072 -> 768 density 0.5, 101 tokens 23 -> 8.7.
//   bf16 768 -> 3072 density 0.5, 2317 tokens 48 -> 22;  4096 -> 4096 density 0.25, 509 tokens 38 -> 29, 64 tokens 21 -> 8.3.
#pragma once
#include <type_traits>

#include "pbs_common.h"
#include "pbs_stream.h"

namespace pbs {

constexpr int ROW_SIZES = 6;    // lists of units: of at most 1, 2, ... 6 blocks
constexpr int ROW_NB = 4;       // sdd_split_kernel has registers for this many, and chunks of 4 GB take this list
constexpr int ROW_NW = 4;       // waves of a workgroup: every ROW_NW-th chunk of tokens each
constexpr int ROW_TC = 32;      // tokens per chunk
constexpr int ROW_GROUP = 8;    // fp32, longer shares: chunks of a wave that are summed before they join its total
constexpr int ROW_LONG = 12, ROW_LONG_GROUPS = 48;   // fp32: chunks of a wave, at most, in units without and with registers for that, other than those of ROW_NB
constexpr int ROW_PARTS = 4;
constexpr int ROW_PIECES = 5;   // LDS of a wave, in pieces of 32 tokens x 32 features

// ---- unit table: what the workgroups of a pattern do ----
// A unit is up to P blocks of one block row: {row, blocks, number within the row, 0, columns [6], data blocks [6]} in 16
// ints.  A row of n blocks has ceil(n / P) units of equal size (+- 1), an empty row one without blocks (for the bias
// gradient).  Order: (quarter of the row's units, row, unit): units that run at the same time then read neighbouring columns of
// X from a common L2.  The table starts with the numbers of units of the lists P = 1 .. ROW_SIZES, padded to 16 ints; then the lists, each in
// room for unit_bound units: some 160 bytes per block of the pattern, where one list of four would take 16.  Derived with the lists of both directions in one
// launch, six lists take 1.3 to 1.8 us more than one (768 -> 3072 density 0.5 6.2 -> 7.6 us, 4096 -> 4096 density 0.25 6.5 -> 8.3).
//
// Why several lists: one workgroup per CU takes as long as its unit, one more than there are CUs takes twice as long, and small patterns of large
// units leave most of the chip idle or need several slices of the tokens and their reduction.  The best list and number of slices of 80 problems each are,
// on average, 1.28 (fp32) and 1.14 (bf16) times as fast as units of four in as many slices as is best for those.
constexpr int UNIT_INTS = 16;
constexpr int UNIT_LDS_ROWS = 1024;
constexpr int ROW_FEW_UNITS = 128;
static __host__ __device__ __forceinline__ long long unit_bound(int rows, int nnz, int P) { return (long long)nnz / P + rows; }   // ceil(n / P) <= n / P + 1 - 1 / P
// A table has all lists (only = 0) or one: of more rows than UNIT_LDS_ROWS that of ROW_NB (they fill the chip with any, and tables are mostly rows
// without blocks), and where a call builds the table in its workspace the one that it takes.
static __host__ __device__ __forceinline__ int unit_lists_only(int rows) { return rows <= UNIT_LDS_ROWS ? 0 : ROW_NB; }
static __host__ __device__ __forceinline__ long long units_before(int rows, int nnz, int P, int only) {   // places of the lists before P's
    long long n = 0;
    for (int p = 1; p < P && !only; ++p) n += unit_bound(rows, nnz, p);
    return n;
}
static __host__ __device__ __forceinline__ unsigned unit_grid(int rows, int nnz, int P) { return (unsigned)((unit_bound(rows, nnz, P) + 255) / 256); }
static inline unsigned unit_table_grid(int rows, int nnz, int only) {
    if (only) return unit_grid(rows, nnz, only);
    unsigned n = 0;
    for (int p = 1; p <= ROW_SIZES; ++p) n += unit_grid(rows, nnz, p);
    return n;
}
static inline size_t unit_prefix_bytes(int N) { return N / 32 > UNIT_LDS_ROWS ? ((size_t)ROW_PARTS * (N / 32) + 1) * sizeof(int) : 0; }
static inline size_t unit_lists_ints(int N, int nnz, int only) {
    const int rows = N / 32;
    return 16 + (size_t)(only ? unit_bound(rows, nnz, only) : units_before(rows, nnz, ROW_SIZES + 1, 0)) * UNIT_INTS;
}
static inline size_t unit_table_bytes(int N, int nnz, int only) { return unit_lists_ints(N, nnz, only) * sizeof(int) + unit_prefix_bytes(N); }
static __device__ __forceinline__ int row_entries(const int32_t* __restrict__ ptr, int nnz, int r, int* lo) {
    const int a = clamp_entry(ptr[r], nnz), b = clamp_entry(ptr[r + 1], nnz);
    *lo = a;
    return b > a ? b - a : 0;
}
static __device__ __forceinline__ int row_units(int n, int P) { return n > 0 ? (n + P - 1) / P : 1; }
static __device__ __forceinline__ int part_lo(int nu, int h) { return (h * nu + ROW_PARTS - 1) / ROW_PARTS; }   // first unit of quarter h
static __device__ __forceinline__ int unit_entry(int n, int nu, int j) { return (int)((long long)n * j / nu); }

// units of list P before (quarter, row), into before [ROW_PARTS * rows + 1]; all threads of the workgroup
template <int NT>
static __device__ void unit_prefix(const int32_t* __restrict__ ptr, int nnz, int rows, int P, int* before, int* s_wave) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int carry = 0;
    for (int base = 0; base < ROW_PARTS * rows; base += NT) {
        const int i = base + tid;
        int v = 0, lo;
        if (i < ROW_PARTS * rows) {
            const int h = i / rows, nu = row_units(row_entries(ptr, nnz, i - h * rows, &lo), P);
            v = part_lo(nu, h + 1) - part_lo(nu, h);
        }
        int incl = v;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(incl, d, 64);
            if (lane >= d) incl += o;
        }
        __syncthreads();
        if (lane == 63) s_wave[wave] = incl;
        __syncthreads();
        int add = carry;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) {
            if (w < wave) add += s_wave[w];
            carry += s_wave[w];
        }
        if (i < ROW_PARTS * rows) before[i] = add + incl - v;
    }
    if (tid == 0) before[ROW_PARTS * rows] = carry;
    __threadfence_block();
    __syncthreads();
}
__global__ __launch_bounds__(1024) void unit_prefix_kernel(const int32_t* __restrict__ ptr, int nnz, int rows, int P, int* before) {
    __shared__ int s_wave[16];
    unit_prefix<1024>(ptr, nnz, rows, P, before, s_wave);
}
struct UnitArgs {
    const int32_t *ptr, *idx;
    int nnz, rows, cols;
    const int* global_before;   // of unit_prefix_kernel, for patterns whose prefix does not fit LDS
    int only;                   // 0: all lists
    int* table;
};
// one unit per thread; workgroup `block` (256 threads)
static __device__ __forceinline__ void unit_table(const UnitArgs& a, int block) {
    const int32_t* __restrict__ ptr = a.ptr;
    const int32_t* __restrict__ idx = a.idx;
    const int nnz = a.nnz, rows = a.rows, cols = a.cols;
    const int* global_before = a.global_before;
    int P = a.only ? a.only : 1;
    while (!a.only && P < ROW_SIZES && block >= (int)unit_grid(rows, nnz, P)) block -= (int)unit_grid(rows, nnz, P++);
    const int bound = (int)unit_bound(rows, nnz, P);
    int* table = a.table + (size_t)units_before(rows, nnz, P, a.only) * UNIT_INTS;
    __shared__ int s_before[ROW_PARTS * UNIT_LDS_ROWS + 1];
    __shared__ int s_wave[4];
    if (!global_before) unit_prefix<256>(ptr, nnz, rows, P, s_before, s_wave);
    const int* before = global_before ? global_before : s_before;
    const int total = before[ROW_PARTS * rows] < bound ? before[ROW_PARTS * rows] : bound;   // (a corrupt pointer array may ask for more)
    const int u = block * 256 + threadIdx.x;
    if (u == 0) a.table[P - 1] = total;
    if (u >= total) return;
    int lo = 0, hi = ROW_PARTS * rows - 1;   // the place that holds unit u
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (before[mid + 1] <= u) lo = mid + 1; else hi = mid;
    }
    const int h = lo / rows, row = lo - h * rows;
    int first;
    const int n = row_entries(ptr, nnz, row, &first), nu = row_units(n, P);
    const int j0 = part_lo(nu, h), j = j0 + u - before[lo];
    const int e0 = unit_entry(n, nu, j), e1 = unit_entry(n, nu, j + 1);
    int* o = table + 16 + (size_t)u * UNIT_INTS;
    o[0] = row;
    o[1] = e1 - e0;
    o[2] = j;
    o[3] = 0;
#pragma unroll
    for (int b = 0; b < ROW_SIZES; ++b) {
        int c = 0, d = -1;
        if (b < e1 - e0) {
            c = idx[2 * (size_t)(first + e0 + b)];
            d = idx[2 * (size_t)(first + e0 + b) + 1];
            if (c < 0 || c >= cols) c = 0, d = -1;   // (an entry outside the range gets no result)
            d = d < 0 || d >= nnz ? -1 : d;
        }
        o[4 + b] = c;
        o[4 + ROW_SIZES + b] = d;
    }
}
__global__ __launch_bounds__(256) void unit_table_kernel(UnitArgs a) { unit_table(a, blockIdx.x); }

// What a training step derives from a pattern, in one launch: the lists of both directions and the units.  A pattern that
// changes every step derives them every step, and each is a launch that the step's products wait for (3, 3 and 5 us and
// the host's time for each; together they take 6).
struct DeriveArgs {
    ListArgs list[2];
    UnitArgs units;      // table == nullptr: none
    int grid[2];         // workgroups of the lists; the rest make units
};
__global__ __launch_bounds__(256) void derive_kernel(DeriveArgs a) {
    const int b = blockIdx.x;
    if (b < a.grid[0]) list_plan(a.list[0], b, a.grid[0]);
    else if (b < a.grid[0] + a.grid[1]) list_plan(a.list[1], b - a.grid[0], a.grid[1]);
    else unit_table(a.units, b - a.grid[0] - a.grid[1]);
}

struct SddRowArgs {
    const void* g;           // [M, N] grad_output
    const void* x;           // [M, K] input
    const int* units;        // a list of unit_table_kernel's
    const int* count;        // how many it holds
    void* out;               // [nnz*32, 32]
    void* bias_out;          // nullptr or [N]
    float* partial;
    int M, N, K, nnz;
    int slices, chunks_per_slice;   // every unit in this many slices of the tokens
    int chunk0;              // the pass starts here
    bool add;                // fp32: a pass behind the first adds to the sums that are there
};
// What a lane holds of a piece, and the products of two pieces (4 x STEPS matrix instructions).  A lane's accumulators of a block
// are d[a][b][v], column i = COL(q, a, v) of row j = FEAT(r, b): eight consecutive columns per row.
template <typename T>
struct RowFrag;
template <>
struct RowFrag<float> {
    static constexpr int STEPS = 8;
    static constexpr int DMA = 4;          // DMA instructions per piece
    float2 v[STEPS];                       // step s: token 4 s + q, features 2 r and 2 r + 1
    static __device__ __forceinline__ int feature(int r, int a) { return 2 * r + a; }
    static __device__ __forceinline__ int place(int a, int v) { return 2 * v + a; }   // of column i among the eight
    __device__ __forceinline__ void read(const unsigned char* piece, int s, int lane) {
        v[s] = *reinterpret_cast<const float2*>(piece + s * 512 + lane * 8);
    }
    __device__ __forceinline__ void sum(float (&o)[2]) const {   // (in pairs: an eighth of the additions to the running sum)
        static_assert(STEPS == 8, "three levels");
        o[0] += ((v[0].x + v[1].x) + (v[2].x + v[3].x)) + ((v[4].x + v[5].x) + (v[6].x + v[7].x));
        o[1] += ((v[0].y + v[1].y) + (v[2].y + v[3].y)) + ((v[4].y + v[5].y) + (v[6].y + v[7].y));
    }
    static __device__ __forceinline__ void mma(f32x4 (&d)[2][2], const RowFrag& g, const RowFrag& x, int s) {
        d[0][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(g.v[s].x, x.v[s].x, d[0][0], 0, 0, 0);
        d[1][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(g.v[s].y, x.v[s].x, d[1][0], 0, 0, 0);
        d[0][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(g.v[s].x, x.v[s].y, d[0][1], 0, 0, 0);
        d[1][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(g.v[s].y, x.v[s].y, d[1][1], 0, 0, 0);
    }
};
template <>
struct RowFrag<bf16_t> {
    static constexpr int STEPS = 1;
    static constexpr int DMA = 2;
    uint4 v[2];                            // half a: tokens 8 q .. 8 q + 7 of one feature
    static __device__ __forceinline__ int feature(int r, int a) { return 8 * (r >> 2) + 4 * a + (r & 3); }
    static __device__ __forceinline__ int place(int a, int v) { return 4 * a + v; }
    __device__ __forceinline__ void read(const unsigned char* piece, int, int lane) {
        const int r = lane & 15, q = lane >> 4;
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            const unsigned char* p = piece + (8 * q + (r >> 2)) * 64 + (r & 3) * 16 + 8 * a;
            const uint2 lo = tr16_b64(p), hi = tr16_b64(p + 256);
            v[a] = make_uint4(lo.x, lo.y, hi.x, hi.y);
        }
    }
    __device__ __forceinline__ void sum(float (&o)[2]) const {
#pragma unroll
        for (int a = 0; a < 2; ++a)
            for (const uint32_t w : {v[a].x, v[a].y, v[a].z, v[a].w}) o[a] += __uint_as_float(w << 16) + __uint_as_float(w & 0xffff0000u);
    }
    static __device__ __forceinline__ void mma(f32x4 (&d)[2][2], const RowFrag& g, const RowFrag& x, int) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int a = 0; a < 2; ++a)
                d[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, g.v[a]), __builtin_bit_cast(bf16x8, x.v[b]), d[a][b], 0, 0, 0);
    }
};

// sum += v; what the addition cuts off goes into the next one (Kahan's compensated sum).  Of an infinity, or a sum that has become one, nothing finite is cut
// off: inf - inf would make the next sum NaN where a plain one stays infinite.
static __device__ __forceinline__ void add_with_rest(float& sum, float& rest, float v) {
    const float add = v - rest, now = sum + add, left = (now - sum) - add;
    rest = left - left == 0.f ? left : 0.f;
    sum = now;
}

template <typename T>
struct SddRowCfg {
    static constexpr int PIECE = 1024 * Elem<T>::ESZ;
    static constexpr int WAVE_LDS = ROW_PIECES * PIECE;
    static constexpr int RED = ROW_NW * 2 * 4 * 1024 + ROW_NW * 32 * 4;   // the waves' sums of two blocks, and of the bias columns
    static constexpr int LDS = ROW_NW * WAVE_LDS > RED ? ROW_NW * WAVE_LDS : RED;
    static constexpr int WPE = sizeof(T) == 4 ? 2 : 3;   // waves per SIMD: LDS allows the former, registers the latter
};

// The pieces of a matrix of M rows: D DMA instructions of ROWS rows each, zeros for rows behind the last one, so that a matrix's last chunk is one like
// the others.  (Loaded by itself behind the loop, one piece after the other and in bf16 two bytes at a time, it cost a workgroup 1 to 6 us: bf16 768 -> 3072
// density 0.5, 2317 tokens 32.7 -> 28.2, 140 tokens 9.3 -> 5.8; 768 -> 768, 1037 tokens 14.95 -> 9.35, fp32 14.9 -> 13.7; 448 -> 2080 density 0.62, 9336 tokens, in
// sdd_split_kernel 104 -> 98.  Whole token counts the same to within 1 %.)
// A chunk is one buffer, and offsets in it are 32-bit numbers.  FAR: chunks of 4 GB and more; lanes have addresses of their own, those behind the last row that of zeros.
static __device__ const uint4 g_zeros = {0, 0, 0, 0};
template <bool FAR, int D, int ROWS>
struct RowSource {
    const unsigned char* base;
    size_t stride;
    int M;
    unsigned voff[D];
    __device__ __forceinline__ RowSource(const unsigned char* base, size_t stride, int M, int row, int place) : base(base), stride(stride), M(M) {
#pragma unroll
        for (int i = 0; i < D; ++i) voff[i] = (unsigned)(i * ROWS + row) * (unsigned)stride + place * 16;
    }
    __device__ __forceinline__ void dma(unsigned lds, int chunk, size_t column_bytes, int i) const {
        const int t0 = chunk * ROW_TC, left = M - t0 < ROW_TC ? M - t0 : ROW_TC;
        dma16_bounded(lds, bounded_buffer(base + (size_t)t0 * stride, (unsigned)left * (unsigned)stride), voff[i] + (unsigned)column_bytes);
    }
};
template <int D, int ROWS>
struct RowSource<true, D, ROWS> {
    const unsigned char* base;
    size_t stride;
    int M;
    __device__ __forceinline__ RowSource(const unsigned char* base, size_t stride, int M, int, int) : base(base), stride(stride), M(M) {}
    __device__ __forceinline__ void dma(unsigned lds, int chunk, size_t column_bytes, int i) const {
        constexpr int CPR = 64 / ROWS;
        const int lane = lane_now();   // (addresses kept over the loop would be spilled)
        const int t = chunk * ROW_TC + i * ROWS + lane / CPR;
        dma16_lanes(lds, t < M ? base + (size_t)t * stride + column_bytes + lane % CPR * 16 : reinterpret_cast<const unsigned char*>(&g_zeros));
    }
};

// Chunks c_lo .. c_hi - 1 of a unit of NB blocks.
template <typename T, int NB, bool FAR>
static __device__ __forceinline__ void sdd_row_body(const SddRowArgs& a, const int* __restrict__ unit, int c_lo, int c_hi, float* partial,
                                                    unsigned char* smem, int lane, int wave) {
    using E = Elem<T>;
    using F = RowFrag<T>;
    using C = SddRowCfg<T>;
    constexpr int ESZ = E::ESZ, PIECE = C::PIECE, D = F::DMA, CPR = 32 * ESZ / 16, RPI = 64 / CPR;
    constexpr int NBX = NB > 0 ? NB : 1;
    const int r = lane & 15, q = lane >> 4;
    const int row = unit[0];
    int cblk[NBX], bblk[NBX];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        cblk[b] = unit[4 + b];
        bblk[b] = unit[4 + ROW_SIZES + b];
    }
    const bool sums = a.bias_out && unit[2] == 0;

    const size_t gs = (size_t)a.N * ESZ, xs = (size_t)a.K * ESZ;   // row strides
    const unsigned char* G = static_cast<const unsigned char*>(a.g) + (size_t)row * (32 * ESZ);
    const unsigned char* X = static_cast<const unsigned char*>(a.x);
    // A wave's LDS: one G piece and the rest X pieces in turn; one or two blocks per row need their G pieces faster and
    // have two of them.
    constexpr int GS = NB == 1 || NB == 2 ? 2 : 1, XS = ROW_PIECES - GS;
    unsigned char* mem = smem + wave * C::WAVE_LDS;
    const unsigned lds = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)mem);
    // DMA instruction i of a piece: tokens RPI i + lane / CPR, 16 bytes per lane; zeros for tokens behind the matrix's last one
    RowSource<FAR, D, RPI> from_g(G, gs, a.M, lane / CPR, lane % CPR), from_x(X, xs, a.M, lane / CPR, lane % CPR);
    auto dma_g = [&](int slot, int chunk, int i) __attribute__((always_inline)) { from_g.dma(lds + slot * PIECE + i * 1024, chunk, 0, i); };
    auto dma_x = [&](int slot, int chunk, int c, int i) __attribute__((always_inline)) {
        from_x.dma(lds + (GS + slot) * PIECE + i * 1024, chunk, (size_t)c * (32 * ESZ), i);
    };

    f32x4 acc[NBX][2][2];
#pragma unroll
    for (int b = 0; b < NBX; ++b)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[b][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    float bsum[2] = {0.f, 0.f};
    // fp32: a chunk's products are summed by themselves and added to the block's total: the error against 64 bits falls from 3.4e-7
    // to 1.3e-7 at 768 -> 3072 with 4096 tokens (one long chain of matrix instructions per wave before), for 1 to 2 % of a training step;
    // each block's addition runs under the products of the next one
    constexpr bool TOTALS = ESZ == 4 && NB > 0;
    f32x4 total[TOTALS ? NBX : 1][2][2];
    // and the totals of ROW_GROUP chunks to those of the wave's share: the roundings of a chain of n additions grow with n, those of both levels with
    // ROW_GROUP + n / ROW_GROUP.  (So that units in few slices have no larger error than those in many: 6984 tokens 704 -> 2720 density 0.106, 55 chunks a wave in
    // place of 19, 1.35e-7 -> 1.76e-7 without, 1.34e-7 with; 1 to 2 % of the time.)  Not in shares of at most ROW_LONG chunks, and units of five and six blocks, which
    // have no registers for it, have no longer ones.
    constexpr bool GROUPS = TOTALS && NB <= ROW_NB;
    f32x4 grand[GROUPS ? NBX : 1][2][2];
    float bleft[2] = {0.f, 0.f};   // (the bias sums, two values a lane, carry what each addition has cut off)
    auto fold = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                total[TOTALS ? b : 0][i][j] += acc[b][i][j];
                acc[b][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
    };
    if constexpr (TOTALS) {
#pragma unroll
        for (int b = 0; b < NBX; ++b)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    total[b][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                    if constexpr (GROUPS) grand[b][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
    }
    auto next_group = [&]() __attribute__((always_inline)) {
        if constexpr (GROUPS) {
#pragma unroll
            for (int b = 0; b < NBX; ++b)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        grand[b][i][j] += total[b][i][j];
                        total[b][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                    }
        }
    };
    auto add_bias = [&](const F& g) __attribute__((always_inline)) {
        if constexpr (ESZ == 4) {
            float of_chunk[2] = {0.f, 0.f};
            g.sum(of_chunk);
#pragma unroll
            for (int i = 0; i < 2; ++i) add_with_rest(bsum[i], bleft[i], of_chunk[i]);
        } else {
            g.sum(bsum);
        }
    };

    int chunk = c_lo + wave;
    if (chunk < c_hi) {
        const int last = chunk + (c_hi - 1 - chunk) / ROW_NW * ROW_NW;   // this wave's last chunk
        auto after = [&](int c, int n) { return c + n * ROW_NW <= last ? c + n * ROW_NW : last; };   // (past the end: the last one again)
        F gf, xf;
        // piece k is block k % NB of chunk k / NB
#pragma unroll
        for (int t = 0; t < GS; ++t)
#pragma unroll
            for (int i = 0; i < D; ++i) dma_g(t, after(chunk, t), i);
        if constexpr (NB > 0) {
#pragma unroll
            for (int k = 0; k < XS; ++k)
#pragma unroll
                for (int i = 0; i < D; ++i) dma_x(k, after(chunk, k / NBX), cblk[k % NBX], i);
        }
        wait_dma(NB > 0 ? (XS - 1) * D : 0);
#pragma unroll
        for (int s = 0; s < F::STEPS; ++s) {
            gf.read(mem, s, lane);
            if constexpr (NB > 0) xf.read(mem + GS * PIECE, s, lane);
        }
        int xat = 0, gat = 0;   // slots of the pieces in xf and gf
        int group_end = c_hi - c_lo > ROW_LONG * ROW_NW ? chunk + ROW_GROUP * ROW_NW : c_hi;
        for (;; chunk += ROW_NW) {
            if (GROUPS && chunk >= group_end) {
                next_group();
                group_end += ROW_GROUP * ROW_NW;
            }
            if (sums) add_bias(gf);
            if constexpr (NB == 0) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
                for (int i = 0; i < D; ++i) dma_g(0, after(chunk, 1), i);
                wait_dma(0);
#pragma unroll
                for (int s = 0; s < F::STEPS; ++s) gf.read(mem, s, lane);
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                // Read below: the next block's piece, asked for XS - 1 blocks ago, and in the chunk's last block the next chunk's
                // G piece.  The tables have the number of younger DMA instructions, for the orders of issue below.
                // (From four blocks on it is the two blocks' before, with the G piece if a chunk began in between.)
                constexpr int YOUNGER4[ROW_SIZES + 1][ROW_SIZES] = {{}, {1}, {4, 8}, {8, 12, 5}, {8, 12, 12, 8}, {8, 12, 12, 8, 8}, {8, 12, 12, 8, 8, 8}};
                constexpr int YOUNGER2[ROW_SIZES + 1][ROW_SIZES] = {{}, {2}, {2, 4}, {4, 6, 4}, {4, 6, 6, 4}, {4, 6, 6, 4, 4}, {4, 6, 6, 4, 4, 4}};
                wait_dma(D == 4 ? YOUNGER4[NB][b] : YOUNGER2[NB][b]);
                const int xnext = xat + 1 == XS ? 0 : xat + 1;
                const int kb = (b + XS) % NBX;       // the piece that takes this block's slot
                const int cn = after(chunk, (b + XS) / NBX), gn = after(chunk, GS);
                const int gnext = GS == 2 ? gat ^ 1 : 0;
#pragma unroll
                for (int s = 0; s < F::STEPS; ++s) {
                    F::mma(acc[b], gf, xf, s);
                    if constexpr (TOTALS) {
                        if (NB > 1 && s == 3) fold((b + NBX - 1) % NBX);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (F::STEPS == 8) {
                        // instruction i overwrites what steps 2 i and 2 i + 1 have read: their products are under way
                        if (b == 0 && (s & 1)) dma_g(gat, gn, s >> 1);
                        if (b == 0 ? s > 0 && !(s & 1) : (s & 1)) dma_x(xat, cn, cblk[kb], b == 0 ? s / 2 - 1 : s >> 1);
                        if (b == 0 && s == 7) dma_x(xat, cn, cblk[kb], 3);
                    } else {
#pragma unroll
                        for (int i = 0; i < D; ++i)
                            if (b == 0) dma_g(gat, gn, i);
#pragma unroll
                        for (int i = 0; i < D; ++i) dma_x(xat, cn, cblk[kb], i);
                    }
                    xf.read(mem + (GS + xnext) * PIECE, s, lane);
                    if (b == NB - 1) gf.read(mem + gnext * PIECE, s, lane);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (TOTALS) {
                    if (NB == 1) fold(0);
                }
                xat = xnext;
                if (b == NB - 1) gat = gnext;
            }
            if (chunk >= last) break;
        }
        wait_dma(0);   // the sums below use the same space
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    if constexpr (TOTALS) {
#pragma unroll
        for (int b = 0; b < NBX; ++b)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    acc[b][i][j] += total[b][i][j];
                    if constexpr (GROUPS) acc[b][i][j] += grand[b][i][j];
                }
    }
    // ---- the waves' sums meet in LDS, two blocks at a time: wave 2 k + jj stores rows FEAT(r, jj) of block k ----
    f32x4* red = reinterpret_cast<f32x4*>(smem);
#pragma unroll
    for (int b0 = 0; b0 < NB; b0 += 2) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 2; ++k)
            if (b0 + k < NB)
#pragma unroll
                for (int i = 0; i < 4; ++i) red[((wave * 2 + k) * 4 + i) * 64 + lane] = acc[(b0 + k) % NBX][i >> 1][i & 1];
        __syncthreads();
        const int k = wave >> 1, jj = wave & 1;
        const int at = k == 0 ? bblk[b0] : bblk[(b0 + 1) % NBX];
        if (b0 + k < NB && at >= 0) {
            float v[8];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                f32x4 s = red[(k * 4 + 2 * i + jj) * 64 + lane];
#pragma unroll
                for (int w = 1; w < ROW_NW; ++w) s += red[((w * 2 + k) * 4 + 2 * i + jj) * 64 + lane];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[F::place(i, e)] = s[e];
            }
            const size_t o = (size_t)at * 1024 + F::feature(r, jj) * 32 + 8 * q;
            if (partial || ESZ == 4) {
                float* p = (partial ? partial : static_cast<float*>(a.out)) + o;
                if (ESZ == 4 && a.add) {
                    const float4 lo = reinterpret_cast<const float4*>(p)[0], hi = reinterpret_cast<const float4*>(p)[1];
                    const float w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] += w[e];
                }
                reinterpret_cast<float4*>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
                reinterpret_cast<float4*>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
            } else {
                uint32_t w[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) w[e] = (uint32_t)Elem<bf16_t>::from_f32(v[2 * e]).bits | ((uint32_t)Elem<bf16_t>::from_f32(v[2 * e + 1]).bits << 16);
                *reinterpret_cast<uint4*>(static_cast<uint16_t*>(a.out) + o) = make_uint4(w[0], w[1], w[2], w[3]);
            }
        }
    }
    if (sums) {
        float* s = reinterpret_cast<float*>(smem + ROW_NW * 2 * 4 * 1024);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            bsum[i] += __shfl_xor(bsum[i], 16, 64);
            bsum[i] += __shfl_xor(bsum[i], 32, 64);
            if (lane < 16) s[wave * 32 + F::feature(lane, i)] = bsum[i];
        }
        __syncthreads();
        if (wave == 0 && lane < 32) {
            float v = s[lane];
#pragma unroll
            for (int w = 1; w < ROW_NW; ++w) v += s[w * 32 + lane];
            if constexpr (ESZ == 4) {
                float* p = (partial ? partial + (size_t)a.nnz * 1024 : static_cast<float*>(a.bias_out)) + row * 32 + lane;
                *p = a.add ? *p + v : v;
            } else if (partial) {
                partial[(size_t)a.nnz * 1024 + row * 32 + lane] = v;
            } else {
                static_cast<T*>(a.bias_out)[row * 32 + lane] = E::from_f32(v);
            }
        }
    }
}

// What a workgroup does: a unit, and its chunks of the tokens.
struct RowTask {
    const int* unit;
    int c_lo, c_hi;
    float* partial;
};
static __device__ __forceinline__ bool row_task(const SddRowArgs& a, RowTask& t) {
    // An XCD takes a run of units and goes through them for one token slice after the other.  Few units do not divide by eight well enough:
    // then it takes an eighth of the tasks, ordered by slice (768 x 768 density 0.5, 16384 tokens fp32, 81 units: 93 us in five slices, of 11 units for
    // most XCDs and so 55 tasks for 64 places, 84 in six with 61 tasks; 141 units 77 against 78).
    const int units = *a.count, xcd = blockIdx.x % NUM_XCD, local = blockIdx.x / NUM_XCD;
    int slice, u;
    if (units < ROW_FEW_UNITS) {
        const int tasks = units * a.slices, id = tasks * xcd / NUM_XCD + local;
        if (id >= tasks * (xcd + 1) / NUM_XCD) return false;
        slice = id / units;
        u = id - slice * units;
    } else {
        const int u_lo = (int)((long long)units * xcd / NUM_XCD), n_u = (int)((long long)units * (xcd + 1) / NUM_XCD) - u_lo;
        if (local >= n_u * a.slices) return false;
        slice = local / n_u;
        u = u_lo + local - slice * n_u;
    }
    t.unit = a.units + (size_t)u * UNIT_INTS;
    const int chunks = (a.M + ROW_TC - 1) / ROW_TC;
    t.c_lo = a.chunk0 + slice * a.chunks_per_slice;
    t.c_hi = t.c_lo + a.chunks_per_slice < chunks ? t.c_lo + a.chunks_per_slice : chunks;
    t.partial = a.slices > 1 ? a.partial + (size_t)slice * ((size_t)a.nnz * 1024 + (a.bias_out ? a.N : 0)) : nullptr;
    return true;
}

template <typename T, bool FAR>
__global__ __launch_bounds__(ROW_NW * 64, SddRowCfg<T>::WPE) void sdd_row_kernel(SddRowArgs a) {
    __shared__ __attribute__((aligned(1024))) unsigned char smem[SddRowCfg<T>::LDS];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    RowTask t;
    if (!row_task(a, t)) return;
    switch (t.unit[1]) {
        case 6: if constexpr (!FAR) sdd_row_body<T, 6, FAR>(a, t.unit, t.c_lo, t.c_hi, t.partial, smem, lane, wave); break;
        case 5: if constexpr (!FAR) sdd_row_body<T, 5, FAR>(a, t.unit, t.c_lo, t.c_hi, t.partial, smem, lane, wave); break;
        case 4: sdd_row_body<T, 4, FAR>(a, t.unit, t.c_lo, t.c_hi, t.partial, smem, lane, wave); break;
        case 3: sdd_row_body<T, 3, FAR>(a, t.unit, t.c_lo, t.c_hi, t.partial, smem, lane, wave); break;
        case 2: sdd_row_body<T, 2, FAR>(a, t.unit, t.c_lo, t.c_hi, t.partial, smem, lane, wave); break;
        case 1: sdd_row_body<T, 1, FAR>(a, t.unit, t.c_lo, t.c_hi, t.partial, smem, lane, wave); break;
        default:
            if (a.bias_out) sdd_row_body<T, 0, FAR>(a, t.unit, t.c_lo, t.c_hi, t.partial, smem, lane, wave);
            break;
    }
}

}  // namespace pbs
