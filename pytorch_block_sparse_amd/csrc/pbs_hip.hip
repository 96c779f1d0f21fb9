// C ABI of libpbs_hip.so: argument checks, tile-shape choice and kernel launches.
#include "../../include/pbs_hip.h"

#include <hip/hip_runtime.h>

#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <tuple>

#include "pbs_common.h"
#include "pbs_dds16.h"
#include "pbs_ddsc.h"
#include "pbs_panel.h"
#include "pbs_split.h"
#include "pbs_stream.h"
#include "pbs_walk.h"
#include "pbs_index.h"
#include "pbs_sdd.h"
#include "pbs_sdd_bf16.h"
#include "pbs_sdd_row.h"
#include "pbs_sdd_split.h"

namespace pbs {

static inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Launches a kernel; the call that the triple brackets end in, without the way through the thread's launch configuration and the last error (2.8 us of a
// launch's host time -> 2.6).  An error is returned and does not stay behind for the next runtime call to report.
template <typename... P, typename... A>
static int launch(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream, const A&... args) {
    std::tuple<P...> values{static_cast<P>(args)...};
    const hipError_t e = std::apply([&](P&... v) {
        void* at[] = {&v...};
        return hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, at, lds, stream);
    }, values);
    if (e != hipSuccess) (void)hipGetLastError();
    return (int)e;
}

// What a call's sizes lead to is worked out once for the sizes that a thread has had last: a call asks for the part of the plan, for its workspace and when it is
// launched, and a model's layers come in turn.  (The choice for 1 token 4096 -> 4096 in bf16, made twice a call of 6.5 us, 220 -> 49 ns, most of that reading the
// environment; the weight gradient's for four layers in turn, three times a gradient, 170 -> 12 ns, where one answer was kept.)
struct Sizes {
    long long M;
    int n, k, nnz, what;   // what: all else that the answer follows from
    bool operator==(const Sizes& o) const { return M == o.M && n == o.n && k == o.k && nnz == o.nnz && what == o.what; }
};
template <typename Answer, typename Ask>
static const Answer& answer(const Sizes& s, const Ask& ask) {   // (the type of `ask` tells the questions apart)
    struct Kept {
        bool there = false;
        Sizes sizes;
        Answer answer;
    };
    static thread_local Kept kept[16];
    Kept& at = kept[(unsigned)((((unsigned)s.M * 31u + s.n) * 31u + s.k) * 31u + s.nnz + s.what) * 2654435761u >> 28];
    if (!at.there || !(at.sizes == s)) at = Kept{true, s, ask()};
    return at.answer;
}

// Zero fill as a kernel (callers may capture the stream into a graph).
__global__ __launch_bounds__(256) void fill_zero_kernel(uint32_t* p, size_t nwords) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < nwords) p[i] = 0u;
}

// Kernels that use more than 64 KB of LDS need the limit raised once per device.
template <typename K>
static int raise_lds_limit(K kernel, int bytes, std::atomic<uint64_t>& done) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    const uint64_t bit = 1ull << (dev & 63);
    if (done.load(std::memory_order_acquire) & bit) return 0;
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return (int)e;
    done.fetch_or(bit, std::memory_order_release);
    return 0;
}

struct DdsArgs {
    const void* a;         // [M, K] row-major
    const void* data;      // [nnz*32, 32]
    const int* plan;       // built by pbs_blocksparse_matmul_plan for this pattern and direction
    const void* bias;      // nullptr or [N]
    void* out;             // [M, N] row-major
    int M, N, K, nnz;
};

// ---- plan buffer ----
// [work list, pbs_stream.h][wide plan, pbs_dds16.h][column plan, pbs_ddsc.h], which is what the products read and
// pbs_blocksparse_matmul_plan_part_bytes counts.  pbs_blocksparse_matmul_plan_bytes counts, behind that, what plans held when the first
// area was records for groups of 8 block columns: per width of 8, 7, 6 and 5 a table of the block column in each of a group's 8 places
// (written by pbs_blocksparse_matmul_plan alone; it tells which columns exist), and for the last three an area of records, not
// written any more.
constexpr int PLAN_NWIDTHS = 4;
constexpr int PLAN_WIDTHS[PLAN_NWIDTHS] = {8, 7, 6, 5};
constexpr int PLAN_PLACES = 8;
static inline size_t width_groups(int n, int wi) { return ((size_t)(n / 32) + PLAN_WIDTHS[wi] - 1) / PLAN_WIDTHS[wi]; }
static inline size_t width_bytes(int n, int k, int wi) { return width_groups(n, wi) * ((size_t)k / 32 + 2) * 64; }
static inline size_t slot_table_bytes_w(int n, int wi) { return (width_groups(n, wi) * PLAN_PLACES * sizeof(int) + 63) / 64 * 64; }
static inline size_t list_area_bytes(int n, int k) { return width_bytes(n, k, 0); }   // >= list_plan_bytes(n, k)
static inline size_t wide_plan_bytes(int n, int k) {
    if (k % 64) return 0;
    const size_t groups = ((size_t)(n / 32) + D16_NB - 1) / D16_NB;
    return (groups * dds16_plan_group_ints(k / 32) + D16_SEQ_INTS) * sizeof(int);
}
static inline size_t column_plan_offset(int n, int k) { return list_area_bytes(n, k) + wide_plan_bytes(n, k); }
static inline int column_groups(int n) { return (n / 32 + DC_NB - 1) / DC_NB; }
static inline size_t column_table_bytes(int n) { return ((size_t)column_groups(n) * DC_NB * sizeof(int) + 63) / 64 * 64; }
static inline size_t column_plan_bytes(int n, int k) {
    // k-pairs, and the lists of a group of 16 columns must fit the kernel's LDS area (16 * k / 32 items)
    // (an odd number of k-blocks where no panel kernel holds the whole contraction)
    if (k % 64 && k <= PANEL_MAX_K) return 0;
    if (DC_NB * (k / 32) > DC_ITEMS_LDS) return 0;
    return column_table_bytes(n) + ((size_t)column_groups(n) * ddsc_plan_group_ints(k / 32) + DC_SEQ_INTS) * sizeof(int);
}
static inline size_t part_plan_bytes(int n, int k) { return column_plan_offset(n, k) + column_plan_bytes(n, k); }
static inline size_t slot_table_offset(int n, int k, int wi) {
    size_t off = part_plan_bytes(n, k);
    for (int i = 1; i <= wi; ++i) off += slot_table_bytes_w(n, i - 1) + width_bytes(n, k, i);
    return off;
}
static inline size_t all_plan_bytes(int n, int k) { return slot_table_offset(n, k, PLAN_NWIDTHS - 1) + slot_table_bytes_w(n, PLAN_NWIDTHS - 1); }

// the block column in each of the 8 places of each group, one table per width: every column once, -1 elsewhere
struct SlotTables {
    int* table[PLAN_NWIDTHS];
    int groups[PLAN_NWIDTHS];
};
__global__ __launch_bounds__(256) void slot_tables_kernel(SlotTables t, int nblk_n) {
#pragma unroll
    for (int wi = 0; wi < PLAN_NWIDTHS; ++wi) {
        const int width = PLAN_WIDTHS[wi];
        for (int i = blockIdx.x * 256 + threadIdx.x; i < t.groups[wi] * PLAN_PLACES; i += gridDim.x * 256) {
            const int j = i % PLAN_PLACES, c = i / PLAN_PLACES * width + j;
            t.table[wi][i] = j < width && c < nblk_n ? c : -1;
        }
    }
}

constexpr int D16_TM = 2, D16_RS = 3, D16_RB = 32, D16_NP = 4;
constexpr double DDSC_MIN_BLOCKS_PER_COLUMN = 32.0;
constexpr int DDSC_WIDE_RESULT = 2048;

// Whether the wide kernel serves this problem: k-pairs need k % 64 == 0, the plan records of a group
// must fit in LDS beside the rings, and there must be enough tiles to give every CU one.
static bool wide_kernel_fits(long long M, int n, int k) {
    using C = D16Cfg<D16_TM, D16_RS, D16_RB, D16_NP>;
    if (k % 64) return false;
    const size_t lds = (size_t)C::WORK_BYTES + dds16_plan_group_ints(k / 32) * sizeof(int);
    if (lds > 160 * 1024) return false;
    const long long tiles = ((M + C::BM - 1) / C::BM) * ((n / 32 + D16_NB - 1) / D16_NB);
    return tiles >= 256;
}

template <int TRANS>
static int launch_dds16(const DdsArgs& g, hipStream_t stream) {
    using C = D16Cfg<D16_TM, D16_RS, D16_RB, D16_NP>;
    static std::atomic<uint64_t> done{0};
    auto kernel = dds16_kernel<TRANS, D16_TM, D16_RS, D16_RB, D16_NP>;
    D16Args a;
    a.a = g.a;
    a.data = g.data;
    a.plan = reinterpret_cast<const int*>(reinterpret_cast<const unsigned char*>(g.plan) + list_area_bytes(g.N, g.K));
    a.bias = g.bias;
    a.out = g.out;
    a.M = g.M;
    a.N = g.N;
    a.K = g.K;
    a.nnz = g.nnz;
    a.m_tiles = (g.M + C::BM - 1) / C::BM;
    a.n_groups = (g.N / 32 + D16_NB - 1) / D16_NB;
    a.group_ints = (int)dds16_plan_group_ints(g.K / 32);
    a.seq = a.plan + (size_t)a.n_groups * a.group_ints;
    // about one workgroup per CU, each walking the token tiles p, p + P, ... of its column group
    int P = 256 / a.n_groups;
    if (P < 1) P = 1;
    if (P > a.m_tiles) P = a.m_tiles;
    a.wg_per_group = P;
    a.stream_step = stream_step(P, a.m_tiles);
    const size_t lds = (size_t)C::WORK_BYTES + (size_t)a.group_ints * sizeof(int);
    if (int rc = raise_lds_limit(kernel, 160 * 1024, done)) return rc;
    return launch(kernel, dim3(stream_grid_blocks(P, a.n_groups, 1)), dim3(C::NT), lds, stream, a);
}

// ---- bf16 kernel with one block column per wave ----
constexpr int DDSC_RS = 8;

// PBS_COLUMN_KERNEL = 0: never use it; 1: whenever it can run; unset: where it is the faster one.
static int column_kernel_wish() {
    const char* e = std::getenv("PBS_COLUMN_KERNEL");
    if (!e || !*e) return -1;
    return e[0] == '0' ? 0 : 1;
}

struct ColumnLaunch {
    int m_tiles, n_groups, wg_per_group;
};
static inline ColumnLaunch column_launch(long long M, int n) {
    ColumnLaunch c;
    c.m_tiles = (int)((M + DC_BM - 1) / DC_BM);
    c.n_groups = column_groups(n);
    int P = 256 / c.n_groups;   // about one workgroup per CU, each walking the token tiles p, p + P, ... of its column group
    if (P < 1) P = 1;
    if (P > c.m_tiles) P = c.m_tiles;
    c.wg_per_group = P;
    return c;
}

// Whether that kernel can run this problem at all, and whether it should.  It reads a block's fragments straight
// from global memory, once per token tile, and its cost per block product is a third of the wide kernel's: 20 %
// faster at 32 blocks per column (the 4096 x 4096 layer at density 0.25), 35 % at 64.  Measured over densities
// 0.008 to 1 and results 512 to 4096 wide (16384 tokens): with a result of 2048 columns or more it is also the
// faster one for sparse patterns (4096 x 4096: 6 to 30 % at 1 to 24 blocks per column; 2048 x 2048: level at 2 to 4
// blocks per column, 5 to 13 % from 8), while results of 512 to 1024 columns stay 10 to 30 % faster in the other
// kernels until their columns hold 32 blocks.
static bool column_kernel_runs(long long M, int n, int k, int nnz) {
    if (!column_plan_bytes(n, k) || nnz < 1 || nnz > DC_MAX_BLOCKS || M < 1) return false;
    const ColumnLaunch c = column_launch(M, n);
    const long long tiles_per_wg = (c.m_tiles + c.wg_per_group - 1) / c.wg_per_group;
    return tiles_per_wg * ((k + 32) / 64) < DC_SEQ_INTS;   // (a workgroup's steps are numbered through the table)
}
static bool column_kernel_fits(long long M, int n, int k, int nnz) {
    if (k % 64 || !column_kernel_runs(M, n, k, nnz)) return false;
    const ColumnLaunch c = column_launch(M, n);
    if ((long long)c.m_tiles * c.n_groups < 256) return false;
    const double per_column = (double)nnz / (n / 32);
    if (per_column >= DDSC_MIN_BLOCKS_PER_COLUMN) return true;
    // wide results (at least four groups of 16 block columns): from 16 blocks per column, and from 2 when the contraction
    // is long enough for the ring to fill (16 k-pairs)
    if (n >= DDSC_WIDE_RESULT && per_column >= 16.0) return true;
    return n >= DDSC_WIDE_RESULT && k >= 1024 && per_column >= 2.0;
}

// Whether its copies ask for lines ahead (pbs_ddsc.h): a dense operand of 100 MB and more is taken to be in memory (of 60 products with operands of 12 to 98 MB, three in
// turn, it makes 6 to 9 one to seven hundredths faster and the others up to 9 slower), with four groups of columns to share the asking (with three 0.96 to 1.03, of 76 products
// of up to 48 blocks a column 35 at least 2 % slower) and columns of up to 40 blocks, 48 where every other row begins in the middle of a line (even products of 33 to 40 blocks a column 1.034
// times as fast, with an odd number of k-blocks 1.055, and of 41 to 48 1.05, where an even number is level; of 49 to 64 8 of 38 and 6 of 32 are slower).  250 products of up to 32 blocks a
// column: even ones 1.05 times as fast, with an odd number of k-blocks 1.08, two slower (0.965, 0.975); with Zipf rows 260 others 1.00 (0.91 to 1.09).
static bool touches(long long M, int n, int k, int nnz) {
    return 2.0 * (double)M * k >= 100e6 && column_groups(n) >= 4 && nnz <= (k % 64 ? 48ll : 40ll) * (n / 32);
}
// FM: the blocks are given in fragment order (the forward product's copy) instead of [n][k] as stored
template <bool FM>
static int launch_ddsc(const DdsArgs& g, const void* data_nk, hipStream_t stream) {
    using C = DdscCfg<DDSC_RS>;
    static std::atomic<uint64_t> done{0};
    auto kernel = ddsc_kernel<DDSC_RS, FM>;
    const ColumnLaunch c = column_launch(g.M, g.N);
    DdscArgs a;
    a.a = g.a;
    a.data = data_nk;
    a.plan = reinterpret_cast<const int*>(reinterpret_cast<const unsigned char*>(g.plan) + column_plan_offset(g.N, g.K) +
                                          column_table_bytes(g.N));
    a.bias = g.bias;
    a.out = g.out;
    a.M = g.M;
    a.N = g.N;
    a.K = g.K;
    a.nnz = g.nnz;
    a.m_tiles = c.m_tiles;
    a.n_groups = c.n_groups;
    a.group_ints = (int)ddsc_plan_group_ints(g.K / 32);
    a.seq = a.plan + (size_t)a.n_groups * a.group_ints;
    a.wg_per_group = c.wg_per_group;
    a.stream_step = stream_step(c.wg_per_group, c.m_tiles);
    a.touch = touches(g.M, g.N, g.K, g.nnz);
    if (int rc = raise_lds_limit(kernel, 160 * 1024, done)) return rc;
    return launch(kernel, dim3(stream_grid_blocks(c.wg_per_group, c.n_groups, c.n_groups & 1 ? 1 : 2)), dim3(C::NT), C::LDS_BYTES, stream, a);
}

// ---- one block column per workgroup ----
struct StreamShape {
    int tt, ks;   // token tile 16 * tt, waves per workgroup
};
// The shapes that are built, of the 15 with tt in {1, 2, 4, 8} and ks in {1, 2, 4, 8} that were timed on 140 problems (1 to
// 16384 tokens, 256 to 4096 features, densities 0.05 to 0.75, even and Zipf columns).  In fp32 the number of waves
// follows from the pattern alone, so that a token's result does not depend, to the last bit, on how many tokens share the call (among the
// calls that run here: split_kernel_fits): four from 14
// blocks per column (then within 1 to 4 % of the best on average), two below (within 5 %; four are 6 to 14 % slower there,
// the sum of the waves' parts weighs more).
constexpr StreamShape STREAM_F32[] = {{1, 2}, {2, 2}, {4, 2}, {1, 4}, {2, 4}, {4, 4}};
constexpr StreamShape STREAM_BF16[] = {{1, 4}, {1, 8}, {2, 2}, {2, 4}, {4, 1}, {4, 2}, {4, 4}, {8, 2}};
static int stream_waves_f32(int n, int nnz) { return (double)nnz / (n / 32) >= 14.0 ? 4 : 2; }

// Estimated time of a shape in us: workgroups per CU x (what a block costs a CU that is kept busy, and what a workgroup
// costs apart from its blocks), plus one workgroup's own chain (launch, list, first operands; then its blocks one after
// the other).  The constants were fitted to the timings above, which they meet within 9 % (bf16) and 11 % (fp32); the
// choice they make is 1.5 % (fp32) and 6 % (bf16) slower than the best built shape on average.  0.0589 us per 16 tokens
// and block is close to the matrix instructions' own rate in fp32.  bf16 tiles of 128 tokens leave a CU one tile at most
// times, so short columns, whose start and end weigh more, do not take them (from 12 blocks per column they are 10 to 20 % faster).
static double stream_us(int esz, long long M, int n, int nnz, StreamShape s) {
    const double cols = n / 32, c = nnz / cols, tt = s.tt, ks = s.ks;
    const double per_cu = (double)((M + 16 * s.tt - 1) / (16 * s.tt)) * cols / 256.0;
    if (esz == 4)
        return std::ceil(per_cu) * (c * (0.0589 * tt + 0.0058) + 0.0976 * tt + 0.0819 * ks) + 3.6 + std::ceil(std::ceil(c) / ks) * 0.235 * tt;
    const double rounds = 0.7 * per_cu + 0.3 * std::ceil(per_cu);
    const double t = rounds * (c * (0.0177 * tt + 0.0067) + 0.0344 * tt + 0.0638 * ks) + 3.8 + std::ceil(std::ceil(c) / ks) * (0.12 + 0.0196 * tt);
    return s.tt == 8 && c < 12.0 ? 2.0 * t : t;
}
struct StreamChoice {
    StreamShape shape;
    double us;
};
static StreamChoice choose_stream_anew(int esz, long long M, int n, int k, int nnz) {
    StreamChoice best{{0, 0}, -1.0};
    auto consider = [&](StreamShape s) {
        // a lane's offset into its token tile is a 32-bit number
        if (16ll * s.tt * k * esz > 0xffffffffll) return;
        const double us = stream_us(esz, M, n, nnz, s);
        if (best.us < 0 || us < best.us) best = StreamChoice{s, us};
    };
    if (esz == 4)
        for (const StreamShape& s : STREAM_F32) {
            if (s.ks == stream_waves_f32(n, nnz)) consider(s);
        }
    else
        for (const StreamShape& s : STREAM_BF16) consider(s);
    return best;
}
static StreamChoice choose_stream(int esz, long long M, int n, int k, int nnz) {
    return answer<StreamChoice>(Sizes{M, n, k, nnz, esz}, [&] { return choose_stream_anew(esz, M, n, k, nnz); });
}

// How a launch goes over the chip.  The 8 XCDs as xcd_t ranges of token tiles x 8 / xcd_t sets of columns (every 8 / xcd_t-th of the ranking, so the sets
// are equally heavy): the split that gives the fullest XCD the fewest workgroups, and of those within 3 % of it the one
// with the least to read per XCD.
struct StreamGrid {
    int m_tiles, xcd_t, group;
    long long grid;
};
static StreamGrid stream_grid(int esz, int tt, long long M, int n, int k, int nnz) {
    return answer<StreamGrid>(Sizes{M, n, k, nnz, esz * 16 + tt}, [&] {
        StreamGrid a;
        a.m_tiles = (int)((M + 16 * tt - 1) / (16 * tt));
        const int cols = n / 32;
        const double tile_bytes = 16.0 * tt * k * esz, col_bytes = 1024.0 * esz * nnz / cols;
        long long fewest = 1ll << 62;
        double least = 0.0;
        a.xcd_t = 1;
        for (int pass = 0; pass < 2; ++pass) {
            for (int t = 1; t <= NUM_XCD; t *= 2) {
                const long long tiles = (a.m_tiles + t - 1) / t, sets = (cols + NUM_XCD / t - 1) / (NUM_XCD / t);
                if (pass == 0) {
                    if (tiles * sets < fewest) fewest = tiles * sets;
                } else if (tiles * sets <= fewest + fewest / 32) {
                    const double bytes = tiles * tile_bytes + sets * col_bytes;
                    if (least == 0.0 || bytes < least) {
                        least = bytes;
                        a.xcd_t = t;
                    }
                }
            }
        }
        // as many token tiles to a pass over the columns as an XCD's L2 (4 MB) holds, at least one
        const double fit = 4e6 / tile_bytes;
        a.group = fit < 1.0 ? 1 : (fit > a.m_tiles ? a.m_tiles : (int)fit);
        a.grid = NUM_XCD * (((long long)a.m_tiles + a.xcd_t - 1) / a.xcd_t) * ((cols + NUM_XCD / a.xcd_t - 1) / (NUM_XCD / a.xcd_t));
        return a;
    });
}

static StreamArgs stream_args(const DdsArgs& g, const StreamGrid& at) { return {g.a, g.data, g.plan, g.bias, g.out, g.M, g.N, g.K, at.m_tiles, at.xcd_t, at.group}; }

template <typename T, int TRANS, int TT, int KS>
static int launch_stream_shape(const DdsArgs& g, hipStream_t stream) {
    constexpr int WPE = TT == 8 ? 2 : (TT == 4 ? 3 : 4);   // waves per SIMD that the registers have to allow
    const StreamGrid at = stream_grid(sizeof(T), TT, g.M, g.N, g.K, g.nnz);
    if (at.grid > (1ll << 30)) return PBS_ERR_TOO_LARGE;
    return launch((stream_kernel<T, TRANS, TT, KS, WPE>), dim3((unsigned)at.grid), dim3(KS * 64), 0, stream, stream_args(g, at));
}

// fp32 with enough token tiles and short columns: whether walk_kernel takes it from stream_kernel.  The estimate: launch, the blocks of the fullest
// CU, a wave's own chain, memory; fitted to 222 products (256 to 4096 features, 600 to 16384 tokens, densities 0.05 to 0.75) within 8 % on average.  It has to be a
// fourteenth below stream_kernel's, from 10 us on, where that would take tiles of 64 tokens (against its tiles of 32 it is 0.92 to 1.08 times as fast).
// How uneven columns are is not known here, and a wave multiplies a column alone: so a contraction has at most 32 blocks, and a full column of them takes at most 0.65 of the launch (a
// wave's block takes half a microsecond).  Of products drawn from those that are taken 300 with even columns are 1.14 times as fast on average, none slower, and 250 with Zipf rows 1.11 times, four
// slower (0.93).  With full columns of 0.65 to 1 of the launch 8 of 15 with Zipf rows were slower, down to 0.73 (922 tokens 672 -> 2656 density 0.14 11.7 -> 18.0 us), and with contractions of 1056 to 2048 features
// 11 of 49 (4893 tokens 1184 -> 3456 density 0.19 76 -> 104), where even ones would gain 1.08.
constexpr double WALK_MARGIN = 0.93, WALK_LEAST = 10.0, WALK_BLOCK = 0.5, WALK_FULL = 0.65;
static bool choose_walk(long long M, int n, int k, int nnz) {
    return answer<bool>(Sizes{M, n, k, nnz, 0}, [&] {
        const StreamChoice stream = choose_stream(4, M, n, k, nnz);
        if (stream.us < WALK_LEAST || stream.shape.tt != 4 || stream.shape.ks != 2 || k > WALK_MAX_K) return false;
        const StreamGrid at = stream_grid(4, WALK_TT, M, n, k, nnz);
        const double blocks = (double)nnz / (n / 32), per_cu = std::ceil((double)at.m_tiles * (n / 32) / 256.0);
        const double t = 3.6 + per_cu * (0.122 * blocks + 0.136) + 0.493 * (std::ceil(blocks) + 1.0) + 0.0712e-6 * (double)M * ((double)n + k);
        return t < WALK_MARGIN * stream.us && WALK_BLOCK * (k / 32) <= WALK_FULL * t && at.grid <= (1ll << 30);
    });
}

template <typename T, int TRANS>
static int launch_stream(const DdsArgs& g, hipStream_t stream) {
    if constexpr (sizeof(T) == 4) {
        if (choose_walk(g.M, g.N, g.K, g.nnz)) {
            const StreamGrid at = stream_grid(4, WALK_TT, g.M, g.N, g.K, g.nnz);
            return launch(walk_kernel<TRANS>, dim3((unsigned)at.grid), dim3(64), 0, stream, stream_args(g, at));
        }
    }
    const StreamShape s = choose_stream(sizeof(T), g.M, g.N, g.K, g.nnz).shape;
#define PBS_STREAM(TT, KS) \
    if (s.tt == TT && s.ks == KS) return launch_stream_shape<T, TRANS, TT, KS>(g, stream);
    PBS_STREAM(1, 4) PBS_STREAM(2, 2) PBS_STREAM(2, 4) PBS_STREAM(4, 2) PBS_STREAM(4, 4)
    if constexpr (sizeof(T) == 4) {
        PBS_STREAM(1, 2)
    } else {
        PBS_STREAM(1, 8) PBS_STREAM(4, 1) PBS_STREAM(8, 2)
    }
#undef PBS_STREAM
    return PBS_ERR_TOO_LARGE;
}

// ---- bf16, the token tile in LDS ----
// Estimated time in us and the number of workgroups per token tile: launch; per round of workgroups over the chip (one per CU) its
// start, the tile, the blocks of the wave with the most, the stores; and what memory takes for the dense operands.  Fitted to 90
// problems (K 256 to 1024, results 256 to 4096 wide, 200 to 16384 tokens, densities 0.1 to 0.75, 1 to 16 workgroups per tile),
// met within 6 % on average; the number it picks is never more than 1.2 % slower than the best one.
struct PanelChoice {
    int splits;   // 0: the kernel cannot run the problem
    double us;
    int turns;    // columns of a wave
    int ways;     // 0: the whole contraction in LDS; else panel_chunk_kernel with so many waves per column
};
static PanelChoice choose_panel(long long M, int n, int k, int nnz) {
    PanelChoice best{0, 0.0, 0, 0};
    const int cols = n / 32;
    // (with fewer columns than waves the estimates would take 17 of 108 products, 0.75 to 1.3 times as fast, 0.97 on average; below 1024 tokens only in chunks, from 768 on where a contraction of 2048 and 48 columns of 16
    // blocks leave the stream kernel more to copy than two workgroups per CU take: 2720 -> 4064 density 0.5, 1015 tokens 31 -> 23 us, 2784 -> 3808 density 0.29, 954 tokens 22.5 -> 18)
    if (nnz < 1 || cols < PANEL_NW || (M < 1024 && (M < 768 || k < 2048 || cols < 48 || nnz < 16 * cols))) return best;
    const double tiles = (double)((M + 16 * PANEL_TT - 1) / (16 * PANEL_TT));
    if (k > PANEL_MAX_K) {
        if (nnz < 5 * cols) return best;   // (shorter columns pay for chunks they do not use: 4 to 13 % slower than the stream kernel at 3 to 4 blocks)
        // the same in chunks, fitted to 90 problems (K 1056 to 4096, results 512 to 4096 wide, 509 to 16384 tokens, densities 0.08 to
        // 0.75; within 9 % on average, its number of waves per column at most 9 % slower than the best): rounds x (start, chunks,
        // blocks of a wave, which a full chip slows down), memory, and the tile once per workgroup that shares it
        for (int ways = 4; ways >= 1; ways /= 2) {
            const int s = (cols + PANEL_NW / ways - 1) / (PANEL_NW / ways);
            const double wgs = tiles * s, full = wgs < 256 ? wgs / 256 : 1.0;
            const double us = 1.68 + std::ceil(wgs / 256) * (1.17 + 0.814 * ((k + PANEL_KC - 1) / PANEL_KC) + (0.359 + 0.221 * full) * nnz / cols / ways) +
                              1e-6 * 2.0 * (double)M * (0.0283 * (n + k) + 0.1363 / 8 * k * s);
            if (best.splits == 0 || us < best.us) best = PanelChoice{s, us, 1, ways};
        }
        return best;
    }
    for (int s = 1; s <= 16 && s <= cols; ++s) {
        const int mine = (cols + s - 1) / s, turns = (mine + PANEL_NW - 1) / PANEL_NW;
        const double us = 2.13 + std::ceil(tiles * s / 256) * (0.656 + 0.051 * (k / 32) + 0.33 * turns * nnz / cols + 0.133 * mine) +
                          0.09e-6 * 2.0 * (double)M * (n + k);
        if (best.splits == 0 || us < best.us) best = PanelChoice{s, us, turns, 0};
    }
    return best;
}
template <int TRANS>
static int launch_panel(const DdsArgs& g, int splits, hipStream_t stream) {
    static std::atomic<uint64_t> done{0};
    auto kernel = panel_kernel<TRANS>;
    const PanelArgs a{g.a, g.data, g.plan, g.bias, g.out, g.M, g.N, g.K, splits};
    const long long wgs = (long long)((g.M + 16 * PANEL_TT - 1) / (16 * PANEL_TT)) * splits;
    if (wgs > (1ll << 30)) return PBS_ERR_TOO_LARGE;
    if (int rc = raise_lds_limit(kernel, 160 * 1024, done)) return rc;
    return launch(kernel, dim3(xcd_grid((int)wgs)), dim3(PANEL_NW * 64), panel_lds(g.K), stream, a);
}

template <int TRANS, int S>
static int launch_panel_chunks(const DdsArgs& g, int splits, hipStream_t stream) {
    static std::atomic<uint64_t> done{0};
    auto kernel = panel_chunk_kernel<TRANS, S>;
    const PanelArgs a{g.a, g.data, g.plan, g.bias, g.out, g.M, g.N, g.K, splits};
    const long long wgs = (long long)((g.M + 16 * PANEL_TT - 1) / (16 * PANEL_TT)) * splits;
    if (wgs > (1ll << 30)) return PBS_ERR_TOO_LARGE;
    if (int rc = raise_lds_limit(kernel, 160 * 1024, done)) return rc;
    return launch(kernel, dim3(xcd_grid((int)wgs)), dim3(PANEL_NW * 64), PANEL_CHUNK_LDS, stream, a);
}

// ---- fp32 on the bf16 matrix cores ----
static inline size_t split_workspace_bytes(int nnz) { return (size_t)nnz * SP_BLOCK_BYTES; }
static inline int split_groups(int n) { return (n / 32 + SP_NC - 1) / SP_NC; }   // (the kernel takes up to half as many again where columns are uneven)

// How many tiles of 64 tokens, the rest being low ones of 32: full tiles for as many whole rounds of units over the 256 CUs as is best, low ones
// behind them (which a result's bits do not depend on).  A low unit takes 0.58 to 0.65 of a full one's time.  Against full tiles alone: 264 units
// (4215 tokens 2784 -> 800) 73 -> 60 us, 128 units (512 tokens 4096 -> 4096) 52 -> 44, multiples of 256 the same.
constexpr double SP_LOW = 0.62;
struct SplitTiles {
    int full;
    double rounds;   // of full units over the chip, in time
};
static SplitTiles split_tiles(long long M, int groups) {
    const long long most = M / SP_BM, all = (M + SP_BM - 1) / SP_BM;
    auto rounds = [&](long long full) {
        const long long low = M > full * SP_BM ? (M - full * SP_BM + 31) / 32 : 0;
        const double f = (double)full * groups / 256, l = (double)low * groups / 256;
        // full rounds, then what is left of the full units beside the low ones
        const double whole = std::floor(f), rest = f - whole;
        if (rest == 0.0) return whole + SP_LOW * std::ceil(l);
        const double beside = (1.0 - rest) * std::floor(1.0 / SP_LOW);   // low units that fit beside the rest
        return whole + 1.0 + (l > beside ? SP_LOW * std::ceil(l - beside) : 0.0);
    };
    SplitTiles best{(int)all, rounds(all)};   // (the last one ragged)
    const long long last = most * groups / 256;
    const int window = 2 + groups / 128;   // (fewer full rounds were the best nowhere)
    for (long long r = last > window ? last - window : 0; r <= last; ++r) {
        const long long full = r * 256 / groups;
        if (full <= most && rounds(full) < best.rounds - 1e-9) best = SplitTiles{(int)full, rounds(full)};
    }
    return best;
}

// Estimated time in us with the launch that splits the blocks: launches; splitting; per round of units over the chip what a step of the ring, a wave's
// blocks (slower where the chip is full) and a unit's start and end cost.  Fitted to 821 products (256 to 4096 features, 512 to 16384 tokens, densities 0.2 to
// 0.8, 2^21 to 2^25 tokens x blocks) whose fullest column holds less than 1.7 times the average; within 5 %.
static double split_us(long long M, int n, int k, int nnz) {
    const int groups = split_groups(n);
    const double units = (double)M / SP_BM * groups / 256, full = units < 1.0 ? units : 1.0;
    return 6.61 + 0.00319 * nnz + split_tiles(M, groups).rounds * (0.101 * (k / 32) + 1.07 * nnz / (n / 32) * (0.669 + 0.331 * full) + 2.48);
}
// Which problems: a density of 0.2 and more, groups of 8 columns that are filled to three quarters, 512 tokens, 4.3 GFLOP (2^21 tokens x blocks), and not
// where the estimates see stream_kernel ahead by a tenth.  Below that density a panel is split for too few products (0.15: 0.8 to 1.1 times as fast, 0.05:
// half as fast); with emptier groups waves have no column; with fewer tokens or products the launch that splits and the first panels weigh too much.
// The tenth is for a result's bits: those of a token are the same, to the last bit, in all calls of a pattern that are served alike, and a line
// at level estimates would part the calls of a 4096 -> 4096 layer of density 0.25 seven times between 512 and 2177 tokens.  Of the 821 products 802 are taken, 1.28
// times faster on average (706 and 1.31 where the estimate has to be 1.08 below), 24 of them more than 2 % slower, the worst 0.83 times as fast, where
// without the estimates 42 were, down to 0.69 (4096 -> 4096 density 0.25, 512 tokens 45 us in stream_kernel and 48 here, 1024 76 and 66, 1025 82 and 94, 2049 152 and 145).
// Columns that are more uneven than that are not known here: 311 of 312 such products (Zipf rows) are taken, 1.10 times faster on average, but 80 of them more than
// 2 % slower, down to 0.57 times as fast where a full column among short ones meets a single round of units (2186 tokens 3104 -> 1472, 1397 blocks
// 59 -> 105 us).
// (Between 1.5 and 2 2^20 tokens x blocks, what the estimate has an eighth faster is 1.10 times as fast with even columns, 1 of 13 slower, and 0.99 with Zipf rows, 6 of 13
// slower, down to 0.79: which of these a pattern is is not known here.)
// (Of 56 products of 9, 10, 11 and 17 columns the estimate, 9 % long for them, would take 22, 1.14 times as fast.  They stay with the fp32 instructions: results of few
// products, as one value to a token gives them, are up to 1.6e-7 off here and one rounding there.)
constexpr double SPLIT_MARGIN = 0.91;
static bool split_kernel_fits(long long M, int n, int k, int nnz) {
    const long long cols = n / 32, groups = split_groups(n);
    if (5ll * nnz < cols * (k / 32) || 4 * cols < 3 * SP_NC * groups || M < 512 || M * nnz < (1 << 21)) return false;
    // units have 32-bit numbers; the waves that wait for one that multiplies a column again (a microsecond per block) must not give up
    if (k > (1 << 16) || (M + 31) / 32 * groups >= (1 << 28)) return false;
    return answer<bool>(Sizes{M, n, k, nnz, 0}, [&] { return SPLIT_MARGIN * split_us(M, n, k, nnz) < choose_stream(4, M, n, k, nnz).us; });
}

// `parts_ready`: the workspace holds the blocks in parts already
template <int TRANS>
static int launch_split(const DdsArgs& g, void* workspace, bool parts_ready, hipStream_t stream) {
    static std::atomic<uint64_t> done{0};
    auto kernel = split_kernel<TRANS>;
    if (int rc = raise_lds_limit(kernel, 160 * 1024, done)) return rc;
    if (!parts_ready)
        if (int rc = launch(split_blocks_kernel<TRANS>, dim3(split_blocks_grid(g.nnz)), dim3(256), 0, stream, static_cast<const float*>(g.data),
                            static_cast<unsigned char*>(workspace), g.nnz)) return rc;
    SplitArgs a;
    a.a = static_cast<const float*>(g.a);
    a.data = static_cast<const float*>(g.data);
    a.parts = static_cast<const unsigned char*>(workspace);
    a.plan = g.plan;
    a.bias = static_cast<const float*>(g.bias);
    a.out = static_cast<float*>(g.out);
    a.M = g.M;
    a.N = g.N;
    a.K = g.K;
    const int groups_even = split_groups(g.N);
    a.heavy = (int)(2ll * g.nnz / (g.N / 32));
    long long units = 0;   // at most
    for (int more = 0; more <= SP_MORE; ++more) {
        a.tiles[more] = split_tiles(g.M, groups_even + more).full;
        const long long low = g.M > (long long)a.tiles[more] * SP_BM ? (g.M - (long long)a.tiles[more] * SP_BM + SP_BM / 2 - 1) / (SP_BM / 2) : 0;
        if (a.tiles[more] + low > units) units = a.tiles[more] + low;
    }
    units *= groups_even + groups_even / 2 + 1;
    // the 32 workgroups of an XCD work on tile_block token tiles x 32 / tile_block groups: the split with the least to read per k-block
    const double w_bytes = (double)SP_NC * SP_BLOCK_BYTES * g.nnz / ((double)(g.N / 32) * (g.K / 32)), x_bytes = SP_BM * 128.0;
    double least = 0.0;
    a.tile_block = 1;
    for (int t = 1; t <= 32; t *= 2) {
        const double groups = groups_even < 32 / t ? groups_even : 32 / t, bytes = t * x_bytes + groups * w_bytes;
        if (groups * t >= 32 || t == 1)
            if (least == 0.0 || bytes < least) {
                least = bytes;
                a.tile_block = t;
            }
    }
    // one workgroup per CU; more where each would have more units than it keeps the heads of
    long long per_xcd = (units + NUM_XCD - 1) / NUM_XCD + 1;
    if (per_xcd > 32) per_xcd = per_xcd > 32 * (SP_MAX_UNITS - 1) ? per_xcd / (SP_MAX_UNITS - 1) + 1 : 32;
    return launch(kernel, dim3((unsigned)(NUM_XCD * per_xcd)), dim3((SP_NC + SP_NP) * 64), SP_LDS, stream, a);
}

// ---- which kernel runs a product ----
enum MatmulPart { PART_LIST = PBS_PLAN_LIST, PART_WIDE = PBS_PLAN_WIDE, PART_COLUMN = PBS_PLAN_COLUMN };   // and so which part of the plan it reads

// Estimated times of the two bf16 kernels with shared panels, in us, from the same kind of fit (140 shapes of 768 to 4096
// features, 1024 to 16384 tokens, within 9 % / 8 %): both walk R token tiles per workgroup, of S k-pairs each.
static double wide_us(long long M, int n, int k, int nnz) {
    const long long m_tiles = (M + D16_BM - 1) / D16_BM, groups = (n / 32 + D16_NB - 1) / D16_NB;
    long long P = 256 / groups;
    P = P < 1 ? 1 : (P > m_tiles ? m_tiles : P);
    return 3.7 + (double)((m_tiles + P - 1) / P) * (0.258 * (k / 64) + 1.394 * nnz / (n / 32) + 5.4);
}
static double column_us(long long M, int n, int k, int nnz, bool copy) {
    const ColumnLaunch c = column_launch(M, n);
    return (double)((c.m_tiles + c.wg_per_group - 1) / c.wg_per_group) * (0.262 * (k / 64) + 0.429 * nnz / (n / 32) + 12.2) + (copy ? 0.0031 * nnz : 0.0);
}
// The column kernel's time outside column_kernel_fits, where its workgroups may be few and its k-blocks odd in number: 274 products (448 to 4096 features, 1200 to 16384
// tokens, densities 0.05 to 0.75, both directions) within 6 % on average.
static double column_anywhere_us(long long M, int n, int k, int nnz, bool copy) {
    const ColumnLaunch c = column_launch(M, n);
    const double tiles = (double)c.m_tiles / c.wg_per_group, rounds = 0.72 * std::ceil(tiles) + 0.28 * tiles, full = c.n_groups * c.wg_per_group / 256.0;
    return 10.4 + rounds * ((k + 32) / 64 * (0.214 + 0.0492 * full) + (double)nnz / (n / 32) * (0.341 + 0.318 * full)) + 1e-6 * 0.131 * M * (n + k) +
           (copy ? 4.2 + 0.00054 * nnz : 0.0);
}
// The column kernel where column_kernel_fits: from 8192 tokens against the stream and the wide kernel without further question
// (it is the faster one in nearly all of that range and within a few us in the rest), otherwise the smallest estimate.
// The panel kernel against it: its estimate is up to 25 % short where a wave takes many full columns (the matrix cores, and
// with them the power limit, are then what counts), the column kernel's is 4 us short for few steps and 12 % long for many; so
// corrected, of 135 problems (K 512 to 1024, results 2048 to 4096 wide, densities 0.1 to 0.75, 4096 to 16384 tokens) the panel kernel
// is given those in which it is 1.05 to 2.2 times the faster one, and the densest ones, where it is up to 13 % the slower one, are not.
struct ProductChoice {
    int part;
    PanelChoice panel;   // splits > 0: panel_kernel or panel_chunk_kernel, which read the list plan like stream_kernel
};
constexpr PanelChoice NO_PANEL{0, 0.0, 0, 0};
static ProductChoice choose_product_anew(long long M, int n, int k, int nnz, int transpose, bool with_copy, int wish) {
    constexpr int esz = 2;
    const bool wide = wide_kernel_fits(M, n, k);
    const bool runs = (!transpose || with_copy) && wish != 0 && column_kernel_runs(M, n, k, nnz), column = runs && column_kernel_fits(M, n, k, nnz);
    if (wish == 1 && runs) return {PART_COLUMN, NO_PANEL};
    if (wish == 0 && wide) return {PART_WIDE, NO_PANEL};
    const PanelChoice panel = choose_panel(M, n, k, nnz);
    const double tc = column ? column_us(M, n, k, nnz, transpose != 0) : 1e300;
    const bool panel_first = panel.splits && !panel.ways && (1.0 + 0.03 * panel.turns) * panel.us < 4.0 + 0.88 * tc;
    if (column && M >= 8192 && !panel_first) return {PART_COLUMN, NO_PANEL};
    // (where the estimates are within 6 % of each other panel_kernel was up to 5 % the slower one as often as the faster: 70 drawn
    // problems, of which it takes 20 and is 1.02 to 1.8 times faster in them; panel_chunk_kernel's is up to 15 % short)
    const double tp = panel.splits ? (panel.ways ? 1.1 : 1.06) * panel.us : 1e300;
    const double ts = choose_stream(esz, M, n, k, nnz).us;
    const double tw = wide ? wide_us(M, n, k, nnz) : 1e300;
    // Outside column_kernel_fits, and inside where panel_first has put a panel kernel before it, from 2048 tokens and 1024 features on, where its estimate is below those of
    // the stream and the panel kernels: by a fourteenth, against panel_chunk_kernel by a seventh in input gradients with contractions of up to 1500 features, and by a fifth in forward products of
    // up to 1350 half of whose blocks are there (that kernel's estimate, with its tenth, is up to 15 % long in these).  Not in place of the wide kernel, whose estimate is from before its workgroups were
    // dealt within the XCDs' CUs: three such products were slower, 0.87 to 0.92.
    // Of 200 products drawn from those that a seventh, a fifth of up to 2048 features, and the wide kernel's estimate wherever it is the smallest had left to the others, 39 against
    // stream_kernel are 1.23 times as fast, none slower, against panel_chunk_kernel 100 even ones 1.08 times (four slower, 0.95) and 61 with Zipf rows, of which the host knows nothing, 1.08 times (nine
    // slower, down to 0.87); 200 that the seventh and the fifth leave out now would be 0.99 times as fast (13394 tokens 2720 -> 1728 density 0.32 114 -> 70 us, 4855 tokens 3936 -> 2016
    // density 0.3 input gradient 52 -> 49, 3983 tokens 3648 -> 1568 density 0.33 35 -> 29).
    if (runs && M >= 2048 && k >= 1024) {
        // (an operand of more than 40 MB goes through memory again for the sets of columns that an XCD has of stream_kernel's, which its estimate does not count: 11386 tokens 3808 -> 2720
        // with 7 blocks a column 68 us where it has 48.  So up to 16 % are added to it here: of 90 drawn layers 13 products more are the column kernel's, 1.23 times as fast, none slower: 15003
        // tokens 2016 -> 3936 density 0.09 100 -> 68, 10288 tokens 3808 -> 2944 density 0.09 87 -> 60.  Without a bound 6 of 17 were slower, down to 0.90; panel and wide kernel chosen for it are 0.81 to
        // 1.13 times as fast.)
        const double mb = 2e-6 * (double)M * k, far = ts + (mb > 40.0 ? std::fmin(2.5e-4 * (mb - 40.0) * n, 0.16 * ts) : 0.0);
        const double least = tp < far ? tp : far;
        const bool wide_first = tw < ts && tw < tp, dense = 2ll * nnz >= (long long)(n / 32) * (k / 32);
        const double below = tp >= far ? 0.93 : (!transpose ? (k <= 1500 ? 0.86 : 0.93) : (dense && k <= 1350 ? 0.80 : 0.93));
        if (!wide_first && column_anywhere_us(M, n, k, nnz, transpose != 0) < below * least) return {PART_COLUMN, NO_PANEL};
    }
    if (column && M >= 8192) return {PART_LIST, panel};
    if (tp < ts && tp < tw && tp < tc) return {PART_LIST, panel};
    if (tc < ts && tc < tw) return {PART_COLUMN, NO_PANEL};
    return {tw < ts ? PART_WIDE : PART_LIST, NO_PANEL};
}
static ProductChoice choose_product(int esz, long long M, int n, int k, int nnz, int transpose, bool with_copy) {
    if (esz == 4) return {PART_LIST, NO_PANEL};
    const int wish = column_kernel_wish();
    return answer<ProductChoice>(Sizes{M, n, k, nnz, (transpose ? 1 : 0) | (with_copy ? 2 : 0) | (wish + 1) << 2},
                                 [&] { return choose_product_anew(M, n, k, nnz, transpose, with_copy, wish); });
}

template <typename T, int TRANS>
static int dispatch_dds(const DdsArgs& g, void* workspace, size_t workspace_bytes, hipStream_t stream, bool parts_ready = false) {
    if constexpr (sizeof(T) == 2) {
        const bool copy = workspace && workspace_bytes >= (size_t)g.nnz * 2048 && aligned16(workspace);
        const ProductChoice choice = choose_product(2, g.M, g.N, g.K, g.nnz, !TRANS, copy);
        const int part = choice.part;
        if (part == PART_COLUMN && (reinterpret_cast<uintptr_t>(g.bias) & 3u) == 0) {   // (it reads the bias in words)
            // the kernel wants every block with k along its rows: as stored for TRANS, a transposed copy otherwise
            if constexpr (TRANS) return launch_ddsc<false>(g, g.data, stream);
            if (int rc = launch(transpose_blocks_kernel, dim3((unsigned)((g.nnz + 3) / 4)), dim3(256), 0, stream,
                                static_cast<const uint16_t*>(g.data), static_cast<uint16_t*>(workspace), g.nnz)) return rc;
            return launch_ddsc<true>(g, workspace, stream);
        }
        if (part == PART_WIDE) return launch_dds16<TRANS>(g, stream);
        switch (choice.panel.splits ? choice.panel.ways : -1) {
            case 0: return launch_panel<TRANS>(g, choice.panel.splits, stream);
            case 1: return launch_panel_chunks<TRANS, 1>(g, choice.panel.splits, stream);
            case 2: return launch_panel_chunks<TRANS, 2>(g, choice.panel.splits, stream);
            case 4: return launch_panel_chunks<TRANS, 4>(g, choice.panel.splits, stream);
            default: break;
        }
    }
    if constexpr (sizeof(T) == 4) {
        if (workspace && workspace_bytes >= split_workspace_bytes(g.nnz) && aligned16(workspace) && split_kernel_fits(g.M, g.N, g.K, g.nnz))
            return launch_split<TRANS>(g, workspace, parts_ready, stream);
    }
    return launch_stream<T, TRANS>(g, stream);
}

// ---- sparse-output product ----
// Two kernels: up to four blocks of a block row per workgroup (pbs_sdd_row.h), which serves fp32 altogether and
// bf16 while the operands are small enough, and for large bf16 problems rectangles of 16 x 16 or 8 x 16 block positions
// (pbs_sdd_bf16.h).
struct SddPlan {
    int rows, tiles_r, tiles_c, nsplit, tokens_per_split;   // rows: block rows of a rectangle, 16 or 8 at most
    bool even;                                              // the same number in all bands
};
static SddPlan plan_rectangles(long long M, int N, int K, int rows, int more_r = 0, int more_c = 0) {   // more bands, and rectangles of a band, than there have to be
    constexpr int SC = SddBf16Cfg<16>::SC, TC = SddBf16Cfg<16>::TC;
    SddPlan p;
    p.rows = rows;
    p.even = false;
    p.tiles_r = (N / 32 + rows - 1) / rows + more_r;
    p.tiles_c = (K / 32 + SC - 1) / SC + more_c;
    const long long tiles = (long long)p.tiles_r * p.tiles_c;
    const long long chunks = (M + TC - 1) / TC;
    // Aim at one workgroup per CU and never slightly more (the kernel's registers and LDS allow one
    // workgroup per CU, so 257 workgroups take twice as long as 256); keep at least 8 chunks per slice.
    long long want = 256 / tiles;
    long long cap = chunks / 8;
    if (cap < 1) cap = 1;
    if (want > cap) want = cap;
    if (want < 1) want = 1;
    const long long chunks_per = (chunks + want - 1) / want;
    p.nsplit = (int)((chunks + chunks_per - 1) / chunks_per);
    if (p.nsplit < 1) p.nsplit = 1;
    p.tokens_per_split = (int)(chunks_per * TC);
    return p;
}
// Estimated time in us of units of at most per_unit blocks, in so many slices: launch, reduction of the slices, chunks of a wave of the slowest workgroup, at
// the rate of a wave alone or of a chip that is full in rounds of 256 workgroups.  Fitted to problems of 256 .. 4096 features, 64 .. 16384 tokens, densities
// 0.05 .. 0.75 at six sizes of units and eight numbers of slices (fp32: 80 below 2^22 tokens x blocks, within 9 %; bf16: 80 whose operands have less than 52 MB,
// within 7 %, and 70 with 40 to 260 MB, within 10 %).  The choices it makes are 3 and 1.5 % slower than the best on average, and 1.28 and 1.14 times as fast as units of
// four in the best number of slices that an estimate of those alone made; 4 fp32 ones of the 160 are slower by more than 2 %, one by 13 %.  Drawn anew, with the
// split kernel and the rectangles among the choices: 864 fp32 problems 1.20 times as fast (23 slower by more than 5 %, the worst 0.87), 621 bf16 ones 1.21 (11, 0.79).
// (The number of units follows from the average row, so what looks like a full chip may be one workgroup more than that: for fp32, whose rounds are long, the mean
// of the estimated number and of 4 % more.  The reduction is a launch and an allocation more for the host: 2 (bf16 0.75) us more than the fit has for it.)
// fp32 on the bf16 matrix cores (sdd_split_kernel) where its estimate is the smaller one, from 2^22 tokens x blocks in units of four (2048 -> 2048 density 0.25, 4096 tokens
// 98 -> 86 us, 4096 -> 4096 density 0.25, 16384 tokens 1267 -> 1091), from 2^20 on, with 256 blocks and more, in units of two to four and at most 8 slices: 50 such problems
// 1.09 times as fast as the fp32 kernel in what its own estimate picks (3072 -> 768 with Zipf rows, 4096 tokens 58 -> 49; 768 -> 3072 density 0.5, 1024 tokens 30.7 -> 27.5; up to 1.28).  Of
// fewer blocks the estimates do not tell which is ahead (0.87 to 1.14), nor of more slices; between 2^17 and 2^20 it is 1.5 % the slower one at its best (36 problems, 0.80 to 1.11).
constexpr long long SPLIT_BACK_WORK = 1ll << 20, SPLIT_BACK_LARGE = 1ll << 22;
constexpr int SPLIT_BACK_BLOCKS = 256, SPLIT_BACK_SLICES = 8;
enum RowKernel { ROW_F32, ROW_SPLIT, ROW_BF16 };   // sdd_row_kernel<float>, sdd_split_kernel, sdd_row_kernel<bf16_t>
// workgroups of the fullest XCD
static double row_tasks(double units, int slices) { return units < ROW_FEW_UNITS ? std::ceil(units * slices / NUM_XCD) : std::ceil(units / NUM_XCD) * slices; }
static double row_us(RowKernel kernel, long long M, int N, int K, int nnz, int per_unit, int slices, int passes) {
    const double chunks = (double)((M + ROW_TC - 1) / ROW_TC), wave = std::ceil(chunks / (ROW_NW * slices * (double)passes));
    struct Model {
        double more, launch, reduce, per_slice, alone, alone_row, busy, busy_row, most, whole, start;   // .._row: of a unit, besides its blocks
        double cached, far, per_mb;   // from so many MB of operands on: how much longer the copies of a full chip take per 100 MB, and what a MB takes at least
    };
    const Model m = kernel == ROW_F32 ? Model{1.04, 3.43, 4.82, 0.973, 0.581, 0.113, 0.549, 0.124, 0.340, 0.880, 0.0191, 0.0, 0.0, 0.0}
                                      : Model{1.0, 3.12, 3.5, 1.31, 0.171, 0.179, 0.140, 0.184, 0.272, 1.0, 0.0128, 52.0, 0.473, 0.2335};
    const double rows = N / 32, row = nnz / rows, columns = K / 32;
    const double full = nnz / (double)per_unit + rows * (per_unit - 1) / (2.0 * per_unit) * (1.0 - std::exp(-2.0 * row)), units = full + rows * std::exp(-row);
    const double mean = nnz / full, most = per_unit < columns ? per_unit : columns;   // blocks of a unit
    if (kernel == ROW_SPLIT) {
        if (M * nnz >= SPLIT_BACK_LARGE) {
            // (units of ROW_NB: 60 such problems at ten slice counts, within 10 %, its choices 1.1 % slower than the best on average.  Fitted without a bound, the cost of
            // a slice came out below nothing, and large gradients were cut into too many: 2048 -> 2048 density 0.25, 4096 tokens 102 -> 86 us)
            const double all_units = nnz >= rows ? nnz / (double)ROW_NB + 0.4 * rows : rows * (1.0 - std::exp(-nnz / rows));   // (those with blocks)
            const double blocks = nnz / all_units > 0.5 ? nnz / all_units : 0.5, tasks = row_tasks(all_units, slices);
            const double busy = std::ceil(tasks / 32) * wave * blocks * 0.454, alone = wave * blocks * 0.540;
            return (slices > 1 ? 3.02 : 0.0) + passes * (7.03 + (busy > alone ? busy : alone) + std::ceil(tasks / 64) * 4.5);
        }
        // (units of two to four: 105 problems of 2^20 tokens x blocks and more, at up to ten numbers of slices, within 6 %; its choices are 1.8 % slower than the best on
        // average, in the larger ones 0.1 % more than those above.  A CU has two workgroups at a time: rounds of 64 over an XCD's 32 CUs, of which the last takes less if no CU has two.)
        const double one = wave * (0.341 * most + 0.591), two = wave * (0.792 * mean + 0.737);
        auto all = [&](double tasks) {
            const double whole = std::floor(tasks / 64), rest = tasks - 64 * whole;
            const double rounds = whole * two + (rest == 0.0 ? 0.0 : rest <= 32 || one > two ? one : two), us = 0.595 * rounds + 0.405 * tasks / 64 * two;
            return (us > one ? us : one) + 0.889 * tasks / 64;
        };
        return (slices > 1 ? 2.0 + 0.4 * slices * nnz / 1000.0 + 0.272 * slices : 0.0) +
               passes * (4.66 + 0.5 * (all(row_tasks(units, slices)) + all(row_tasks(1.03 * units, slices))));
    }
    const double tasks = row_tasks(units, slices), tasks_more = m.more > 1.0 ? row_tasks(m.more * units, slices) : tasks;
    const double alone = wave * (m.alone * (mean + m.most * (most - mean)) + m.alone_row);
    const double rounds = 0.5 * (m.whole * (std::ceil(tasks / 32) + std::ceil(tasks_more / 32)) + (1.0 - m.whole) * (tasks + tasks_more) / 32);
    const double mb = 1e-6 * M * ((double)N + K) * (kernel == ROW_BF16 ? 2 : 4), far = mb > m.cached ? 1.0 + m.far * 0.01 * (mb - m.cached) : 1.0, least = mb > m.cached ? m.per_mb * mb : 0.0;
    const double busy = rounds * wave * (m.busy * mean + m.busy_row) * far;
    const double us = busy > alone ? (busy > least ? busy : least) : (alone > least ? alone : least);
    return (slices > 1 ? m.reduce + m.per_slice * slices * nnz / 1000.0 : 0.0) + passes * (m.launch + us + 0.5 * (tasks + tasks_more) * m.start);
}
// Launch; per round of workgroups and chunk what a pass costs and what the blocks of a wave cost; reduction of the slices (75 problems, 256 .. 16384
// tokens, 256 .. 4096 features, densities 0.05 .. 0.95, one in seven with uneven rows: within 11 % for 16 rows and 9 % for 8).
static double rectangle_us(const SddPlan& p, int nnz) {
    using C = SddBf16Cfg<16>;
    const double tiles = (double)p.tiles_r * p.tiles_c, blocks = nnz / tiles;
    const double rounds = std::ceil(tiles * p.nsplit / 256), passes = std::ceil(blocks / C::QMAX), chunks = p.tokens_per_split / C::TC;
    const double reduce = p.nsplit * (nnz / 1000.0);
    if (p.rows == 16) return 9.84 + rounds * (3.57 + chunks * (0.709 * passes + 0.1114 * blocks / 8)) + (p.nsplit > 1 ? 1.20 + 1.15 * reduce : 0.0);
    return 10.1 + rounds * chunks * (0.738 * passes + 0.0713 * blocks / 8) + (p.nsplit > 1 ? 3.20 + 1.24 * reduce : 0.0);
}
// Rectangles of eight block rows read X once per eight rows but need one pass where sixteen rows hold more blocks than the accumulators, and half the
// slices: 4096 -> 4096, 16384 tokens, density 0.25 198 us with sixteen rows and 265 with eight, 0.5 383 and 339; 768 -> 3072 density 0.5 103 and 77.
// Of the 75 problems the estimates pick the faster one or one within 2 %.
static SddPlan plan_small(long long M, int N, int K, int nnz) {
    const SddPlan tall = plan_rectangles(M, N, K, 16), flat = plan_rectangles(M, N, K, 8);
    return rectangle_us(flat, nnz) < rectangle_us(tall, nnz) ? flat : tall;
}
// Operands beyond 52 MB: more rectangles than there have to be where the fullest would hold more blocks than the accumulators.  It takes two passes over its tokens then, and the
// launch waits for it: 77 blocks take 1.4 times as long as 66.  The fullest one: the rows of the largest band, the columns (dealt in pairs by their blocks)
// of the largest rectangle, and 1.6 times the deviation of a band's blocks.  Fitted to 34 problems of 90 MB and more in 16 partitions each, within 6 % on average; the ratio of two
// partitions of a problem, where the blocks of the fullest rectangle are known, within 5 % for 270 of 52 to 260 MB.
// Of 600 problems of 52 MB and more that it partitions in another way than rectangle_us (one in six), the 300 without structure are 1.23 times as fast, 20 of them slower (down to
// 0.85: what is fullest is up to chance), and the 300 with Zipf rows 1.24 times, 20 slower (0.81).  Taken only where the fullest rectangle is likelier to take two passes (1, 0 and -2
// deviations instead of 1.6 for the partition that is left) 13, 5 and 0 of the 300 are slower, but the others gain 1.22, 1.21 and 1.15.
// us: 15343 tokens 1760 -> 2784 density 0.71 249 -> 166, 13000 tokens 2304 -> 2752 density 0.3 140 -> 96, 12000 tokens 3072 -> 3072 density 0.3 153 -> 119,
// 16384 tokens 2048 -> 2048 density 0.6 171 -> 127; 4096 -> 4096 at density 0.25 and 0.5 as before.
static double partition_us(const SddPlan& p, int N, int K, int nnz) {
    using C = SddBf16Cfg<16>;
    const double rows = N / 32, columns = K / 32, row = nnz / rows, density = row / columns;
    const int row_pairs = (N / 32 + 1) / 2, column_pairs = (K / 32 + 1) / 2;
    int band = 2 * ((row_pairs + p.tiles_r - 1) / p.tiles_r);
    if (!p.even || band > p.rows) band = p.rows;
    double share = 2.0 * ((column_pairs + p.tiles_c - 1) / p.tiles_c) / columns;
    if (share > 1.0) share = 1.0;
    const double most = row * band * share + 1.6 * std::sqrt(band * columns * density * (density < 1.0 ? 1.0 - density : 0.0)) / p.tiles_c + 1.0;
    const double passes = std::ceil(most / C::QMAX), rounds = std::ceil((double)p.tiles_r * p.tiles_c * p.nsplit / 256), chunks = p.tokens_per_split / C::TC;
    const double us = p.rows == 16 ? 15.2 + rounds * (8.6 + chunks * (0.806 * passes + 0.053 * most / 8)) : 14.9 + rounds * (8.3 + chunks * (0.77 * passes + 0.027 * most / 8));
    return us + (p.nsplit > 1 ? 2.5 + 0.68 * p.nsplit * (nnz / 1000.0) : 0.0);
}
static SddPlan plan_sdd(long long M, int N, int K, int nnz) {
    SddPlan best = plan_small(M, N, K, nnz);
    if (2.0 * (double)M * ((double)N + K) <= 52e6) return best;
    double least = 0.93 * partition_us(best, N, K, nnz);   // (differences below that are within the estimate)
    for (int rows = 16; rows >= 8; rows -= 8)
        for (int more_r = 0; more_r <= 4; ++more_r)
            for (int more_c = 0; more_c <= 2; ++more_c) {
                SddPlan p = plan_rectangles(M, N, K, rows, more_r, more_c);
                p.even = true;
                const double us = partition_us(p, N, K, nnz);
                if (us < least) {
                    best = p;
                    least = us;
                }
            }
    return best;
}
// The kernel and, for the row kernel, the number of token slices of a launch (0: rectangles) and of launches, one behind the
// other over consecutive ranges of the tokens.
//
// fp32 wants slices of about 64 MB of the operands: workgroups of different rows read the same columns of X and find them in the
// last-level cache while a slice is about that size (4096 -> 4096 density 0.25, 16384 tokens: 1398 us in one slice, 1333 in four,
// 1233 in eight).  But every slice of a launch is a copy of the gradient in the workspace, so a launch has at most as many as
// fit ROW_WORKSPACE_BYTES, and further launches add to the sums that are there.  Slices x launches, us, against eight slices and more
// in one launch (whose workspace is 128 MB for the first and grows with tokens and features): 4096 -> 4096, 16384 tokens, density 0.25
// 4 x 2 1199 against 1222, 0.5 2 x 4 2258 against 2347, 1 1 x 8 4131 against 4297; 65536 tokens, density 1 1 x 33 16538 against
// 16998; 8192 -> 8192, 16384 tokens, density 0.25 1 x 16 4805 against 5211, 0.5 9264 against 10299.
constexpr size_t ROW_WORKSPACE_BYTES = 64u << 20;
// where the input gradient's blocks are split, the launch that adds the slices does it
constexpr double REDUCE_SAVES = 4.0;
// a chunk of 32 tokens that has 4 GB or more: it is not addressed as one buffer
static bool row_far(int esz, int N, int K) { return (long long)(N > K ? N : K) * esz * ROW_TC >= (1ll << 32); }
struct RowChoice {
    int slices, passes, per_unit;
    bool split;
};
static RowChoice choose_row(int dtype, long long M, int N, int K, int nnz, bool lists, size_t workspace_limit) {
    constexpr int CANDIDATES[] = {1, 2, 3, 4, 5, 6, 8, 11, 16, 24};
    const double bytes = (double)M * ((double)N + K) * (dtype == PBS_DTYPE_F32 ? 4 : 2);
    // (rectangles count the bytes of a chunk in 31 bits)
    const bool rectangles = dtype == PBS_DTYPE_BF16 && N < (1 << 25) && K < (1 << 25);
    // bf16 operands beyond the size of the L2s (52 MB): the rectangles read every panel once per 16 or 8 rows of blocks, the units once per block, but only what
    // they need, so below a density of 0.1 (rectangles with less than 26 of 256 places taken) and 90 MB the units are given what their estimate has at least a tenth faster
    // (of such problems with 52 to 88 MB they take 19 that were the rectangles', 1.18 times as fast on average, 2 of them slower (0.91 and 0.96): 8690 tokens 1184 -> 1888 density 0.05
    // 32 -> 24 us.  Of 8 with 97 to 130 MB 3 were slower, 0.96 on average: 12921 tokens 1024 -> 2720 density 0.054 40 -> 55, 10498 tokens 2592 -> 3616 density 0.06 84 -> 109.)
    // Above that density they are 0.55 to 1.5 times as fast (4096 -> 4096 density 0.25, 16384 tokens 250 us and 198), where the estimates are not good enough to choose; and where
    // most rows are empty, units cost what no estimate counts.  What the workspace does not allow the rectangles is refused and not served another way.
    const bool large = rectangles && bytes > 52e6;
    const bool fits = workspace_limit >= ROW_WORKSPACE_BYTES || plan_rectangles(M, N, K, 16).nsplit * (size_t)nnz * 4096 <= workspace_limit;
    if (large && (bytes > 90e6 || 10ll * nnz >= (long long)(N / 32) * (K / 32) || nnz < N / 32 || !fits)) return {0, 1, ROW_NB, false};
    const long long chunks = (M + ROW_TC - 1) / ROW_TC;
    const double at_least = dtype == PBS_DTYPE_F32 ? std::floor(bytes / 64e6) : 1.0;
    RowChoice best{1, 1, ROW_NB, false};
    double best_us = -1.0;
    const double saved = dtype == PBS_DTYPE_F32 && split_kernel_fits(M, K, N, nnz) ? REDUCE_SAVES : 0.0;
    const bool far = row_far(dtype == PBS_DTYPE_F32 ? 4 : 2, N, K), one_list = far || unit_lists_only(N / 32);
    for (const int s : CANDIDATES) {
        if (s > 1 && (s > chunks / 4 || (size_t)nnz * 4096 * s > workspace_limit)) break;
        const int passes = at_least > s ? (int)std::ceil(at_least / s) : 1;
        auto consider = [&](RowKernel kernel, int per_unit) {
            // (a table of larger lists, made in the workspace, takes of the memory of the partial sums: what they and the list of ROW_NB may have stays the bound)
            if (!lists && per_unit != ROW_NB && (s > 1 ? (size_t)nnz * 4096 * s : 0) + unit_table_bytes(N, nnz, per_unit) > workspace_limit + unit_table_bytes(N, nnz, ROW_NB)) return;
            // (fp32: sums of longer shares would be less exact than those of units of four in several slices)
            if (kernel == ROW_F32 && per_unit != ROW_NB && chunks > (long long)(per_unit > ROW_NB ? ROW_LONG : ROW_LONG_GROUPS) * ROW_NW * s * passes) return;
            const double us = row_us(kernel, M, N, K, nnz, per_unit, s, passes) - (s > 1 ? saved : 0.0);
            if (best_us < 0.0 || us < best_us) {
                best = {s, passes, per_unit, kernel == ROW_SPLIT};
                best_us = us;
            }
        };
        for (int p = one_list ? ROW_NB : 1; p <= (one_list ? ROW_NB : ROW_SIZES); ++p) consider(dtype == PBS_DTYPE_F32 ? ROW_F32 : ROW_BF16, p);
        if (dtype == PBS_DTYPE_F32 && !far) {
            if (M * nnz >= SPLIT_BACK_LARGE) consider(ROW_SPLIT, ROW_NB);
            else if (M * nnz >= SPLIT_BACK_WORK && nnz >= SPLIT_BACK_BLOCKS && s <= SPLIT_BACK_SLICES)
                for (int p = one_list ? ROW_NB : 2; p <= ROW_NB; ++p) consider(ROW_SPLIT, p);
        }
    }
    // (of a density below 0.1, and up to 52 MB, the partition is that of plan_small)
    if (rectangles && fits && (large ? 0.9 : 1.0) * rectangle_us(plan_small(M, N, K, nnz), nnz) < best_us) best.slices = 0;
    return best;
}
struct BackPlan {
    int slices;   // row kernel; 0: rectangles
    int per_unit; // blocks of a unit, at most
    bool split;   // fp32 in parts
    int passes, chunks_per_slice;
    SddPlan rect; // of rectangles only
    int partials;            // sums of this many slices in the workspace, or none
    size_t partial_bytes;
};
static BackPlan plan_back_anew(int dtype, long long M, int N, int K, int nnz, bool lists, size_t workspace_limit) {
    BackPlan p{};
    const RowChoice row = choose_row(dtype, M, N, K, nnz, lists, workspace_limit);
    p.slices = row.slices;
    p.per_unit = row.per_unit;
    p.split = row.split;
    int n = 0;
    if (p.slices > 0) {
        const long long chunks = (M + ROW_TC - 1) / ROW_TC, shares = (long long)row.slices * row.passes;
        p.chunks_per_slice = (int)((chunks + shares - 1) / shares);
        const long long filled = (chunks + p.chunks_per_slice - 1) / p.chunks_per_slice;   // slices with tokens
        p.slices = n = (int)(filled < row.slices ? filled : row.slices);
        p.passes = (int)((filled + n - 1) / n);   // (the last launch may have slices without tokens, which add nothing)
    } else {
        p.rect = plan_sdd(M, N, K, nnz);
        // (the workspace of sixteen rows also where eight need less: what an entry point without one refuses does not follow the estimates)
        const int tall = plan_rectangles(M, N, K, 16).nsplit;
        n = tall > p.rect.nsplit ? tall : p.rect.nsplit;
    }
    p.partials = n > 1 ? n : 0;
    return p;
}
// `lists`: the caller brings a table with all lists of units
static BackPlan plan_back(int dtype, long long M, int N, int K, int nnz, bool bias, bool lists, size_t workspace_limit = ROW_WORKSPACE_BYTES) {
    BackPlan p = answer<BackPlan>(Sizes{M, N, K, nnz, dtype | (lists ? 2 : 0) | (int)((ROW_WORKSPACE_BYTES - workspace_limit) / 16) << 2},
                                  [&] { return plan_back_anew(dtype, M, N, K, nnz, lists, workspace_limit); });
    p.partial_bytes = ((size_t)nnz * 1024 + (bias ? N : 0)) * sizeof(float) * p.partials;   // fp32 sums of each slice: blocks, bias columns
    return p;
}

struct BackArgs {
    const void *g, *x;       // [M, N] grad_output, [M, K] input
    const int32_t *ptr, *idx;
    const void* units;       // nullptr: built in the workspace, if it is needed
    bool lists;              // it would have all lists
    void* out;               // [nnz*32, 32]
    void* bias_out;          // nullptr or [N]
    int M, N, K, nnz;
    const void* data;        // nullptr, or blocks that the launch which adds the slices (there has to be one; fp32) writes to `parts` for an input gradient
    void* parts;
};

static int build_units(const int32_t* ptr, const int32_t* idx, int N, int K, int nnz, int only, void* table, hipStream_t stream) {
    int* t = static_cast<int*>(table);
    int* before = nullptr;
    if (unit_prefix_bytes(N)) {
        before = t + unit_lists_ints(N, nnz, only);
        if (int rc = launch(unit_prefix_kernel, dim3(1), dim3(1024), 0, stream, ptr, nnz, N / 32, only, before)) return rc;
    }
    const UnitArgs a{ptr, idx, nnz, N / 32, K / 32, before, only, t};
    return launch(unit_table_kernel, dim3(unit_table_grid(N / 32, nnz, only)), dim3(256), 0, stream, a);
}

template <typename T>
static int launch_reduce(const float* partial, const BackArgs& a, int nsplit, hipStream_t stream) {
    const size_t n = (size_t)a.nnz * 1024, total = n + (a.bias_out ? a.N : 0);
    const unsigned reducing = (unsigned)((total / 4 + 255) / 256);
    if constexpr (sizeof(T) == 4) {
        if (a.data)
            return launch(sdd_reduce_split_kernel, dim3(reducing + split_blocks_grid(a.nnz)), dim3(256), 0, stream, partial, static_cast<float*>(a.out), n,
                          static_cast<float*>(a.bias_out), total, nsplit, reducing, static_cast<const float*>(a.data), static_cast<unsigned char*>(a.parts),
                          a.nnz);
    }
    return launch(sdd_reduce_kernel<T>, dim3(reducing), dim3(256), 0, stream, partial, static_cast<T*>(a.out), n, static_cast<T*>(a.bias_out), total, nsplit);
}

template <typename T>
static int launch_row(const BackArgs& a, const BackPlan& p, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    const int only = a.units ? unit_lists_only(a.N / 32) : p.per_unit;
    const size_t need = p.partial_bytes + (a.units ? 0 : unit_table_bytes(a.N, a.nnz, only));
    if (need > 0 && (!workspace || workspace_bytes < need || !aligned16(workspace))) return PBS_ERR_WORKSPACE;
    const long long grid = NUM_XCD * (long long)p.slices * ((unit_bound(a.N / 32, a.nnz, p.per_unit) + NUM_XCD - 1) / NUM_XCD);
    if (grid > (1ll << 30)) return PBS_ERR_TOO_LARGE;
    SddRowArgs r;
    r.g = a.g;
    r.x = a.x;
    const int* table = static_cast<const int*>(a.units);
    if (!a.units) {
        void* t = static_cast<unsigned char*>(workspace) + p.partial_bytes;
        if (int rc = build_units(a.ptr, a.idx, a.N, a.K, a.nnz, only, t, stream)) return rc;
        table = static_cast<const int*>(t);
    }
    r.count = table + p.per_unit - 1;
    r.units = table + 16 + units_before(a.N / 32, a.nnz, p.per_unit, only) * UNIT_INTS;
    r.out = a.out;
    r.bias_out = a.bias_out;
    r.partial = p.partial_bytes ? static_cast<float*>(workspace) : nullptr;
    r.M = a.M;
    r.N = a.N;
    r.K = a.K;
    r.nnz = a.nnz;
    r.slices = p.slices;
    r.chunks_per_slice = p.chunks_per_slice;
    for (int pass = 0; pass < p.passes; ++pass) {
        r.chunk0 = pass * p.slices * p.chunks_per_slice;
        r.add = pass > 0;
        const auto kernel = sizeof(T) == 4 && p.split ? sdd_split_kernel : (row_far(sizeof(T), a.N, a.K) ? sdd_row_kernel<T, true> : sdd_row_kernel<T, false>);
        if (int rc = launch(kernel, dim3((unsigned)grid), dim3(ROW_NW * 64), 0, stream, r)) return rc;
    }
    return p.partial_bytes ? launch_reduce<T>(r.partial, a, p.slices, stream) : PBS_OK;
}

template <bool BIAS>
static int launch_rectangles(const BackArgs& b, const BackPlan& plan, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    const SddPlan& p = plan.rect;
    SddArgs a;
    a.g = b.g;
    a.x = b.x;
    a.ptr = b.ptr;
    a.idx = b.idx;
    a.out = b.out;
    a.bias_out = b.bias_out;
    a.partial = nullptr;
    a.M = b.M;
    a.N = b.N;
    a.K = b.K;
    a.nnz = b.nnz;
    a.rows = p.rows;
    a.even = p.even;
    // (a column unit more than the others in the largest rectangle, and a block for how they are dealt)
    const double units = (b.K / 32 + 1) / 2, share = std::ceil(units / p.tiles_c) / units, mean = (double)b.nnz / ((double)p.tiles_r * p.tiles_c);
    const double band_room = (std::ceil(mean / SddBf16Cfg<16>::QMAX) * SddBf16Cfg<16>::QMAX - 1.0) / share;
    a.band_room = band_room < 2147483647.0 ? (int)band_room : 2147483647;
    a.tiles_r = p.tiles_r;
    a.tiles_c = p.tiles_c;
    a.nsplit = p.nsplit;
    a.tokens_per_split = p.tokens_per_split;
    if (p.nsplit > 1) {
        if (!workspace || workspace_bytes < plan.partial_bytes || !aligned16(workspace)) return PBS_ERR_WORKSPACE;
        a.partial = static_cast<float*>(workspace);
    }
    const long long wgs = (long long)p.tiles_r * p.tiles_c * p.nsplit;
    if (wgs > (1ll << 30)) return PBS_ERR_TOO_LARGE;
    using C = SddBf16Cfg<16>;   // (the buffers of both)
    static std::atomic<uint64_t> done{0};
    auto kernel = sdd_bf16_kernel<BIAS>;
    if (int rc = raise_lds_limit(kernel, C::LDS_BYTES, done)) return rc;
    if (int rc = launch(kernel, dim3(xcd_grid((int)wgs)), dim3(C::NT), C::LDS_BYTES, stream, a)) return rc;
    return p.nsplit > 1 ? launch_reduce<bf16_t>(a.partial, b, p.nsplit, stream) : PBS_OK;
}

// ---- scratch of the entry point that allocates nothing ----
// One device array per GPU, part of the library's code object: it exists on every GPU the library runs on
// from the moment the code object is loaded there until the process ends.  Host code never uses the
// array's name as an address (on the host it only stands for the symbol): the address on a device is
// asked for once, with that device current, and kept.
static __device__ __align__(256) unsigned char scratch[PBS_NOALLOC_SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
static void* g_scratch_ptr[MAX_DEVICES];
static std::mutex g_scratch_mutex;

static int scratch_of_current_device(void** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= MAX_DEVICES) return PBS_ERR_TOO_LARGE;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return (int)e;
        if (!p) return PBS_ERR_WORKSPACE;
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return PBS_OK;
}

}  // namespace pbs

using namespace pbs;

extern "C" {

int pbs_abi_version(void) { return PBS_ABI_VERSION; }


const char* pbs_error_string(int code) {
    switch (code) {
        case PBS_OK: return "ok";
        case PBS_ERR_NULL_POINTER: return "pbs: null pointer argument";
        case PBS_ERR_BAD_SHAPE: return "pbs: bad shape (negative size, or a feature dimension that is not a multiple of 32)";
        case PBS_ERR_BAD_DTYPE: return "pbs: unknown dtype code";
        case PBS_ERR_MISALIGNED: return "pbs: dense/data pointers must be 16-byte aligned";
        case PBS_ERR_WORKSPACE: return "pbs: workspace missing, misaligned or too small";
        case PBS_ERR_TOO_LARGE: return "pbs: size exceeds the kernels' index range";
        case PBS_ERR_SCRATCH: return "pbs: the problem needs more scratch than the library's built-in buffer holds; use the entry point that takes a workspace";
        default: break;
    }
    if (code > 0) return hipGetErrorString(static_cast<hipError_t>(code));
    return "pbs: unknown error code";
}

int pbs_build_indices(const uint8_t* mask, const int64_t* block_ptr, int X, int Y, int nnz, int32_t* cols_a,
                      int32_t* row_start_ends_a, int32_t* rows_b, int32_t* col_start_ends_b, int32_t* blocks,
                      int32_t* status, void* stream) {
    if (X < 1 || Y < 1 || nnz < 0 || (long long)nnz > (long long)X * Y) return PBS_ERR_BAD_SHAPE;
    if ((long long)X * Y > (1ll << 30)) return PBS_ERR_TOO_LARGE;
    if (!mask || !row_start_ends_a || !col_start_ends_b || !status) return PBS_ERR_NULL_POINTER;
    if (nnz > 0 && (!cols_a || !rows_b || !blocks)) return PBS_ERR_NULL_POINTER;
    return launch(build_indices_kernel, dim3(1), dim3(INDEX_THREADS), 0, static_cast<hipStream_t>(stream), mask,
                  block_ptr, X, Y, nnz, cols_a, row_start_ends_a, rows_b, col_start_ends_b, blocks, status);
}

size_t pbs_replace_blocks_workspace_bytes(int X, int Y, int nnz) {
    return X < 1 || Y < 1 || nnz < 0 ? 0 : replace_ws_bytes(X, Y, nnz);
}

int pbs_replace_blocks(const int32_t* old_blocks, const int64_t* moves, int n_moves, int X, int Y, int nnz, int32_t* cols_a,
                       int32_t* row_start_ends_a, int32_t* rows_b, int32_t* col_start_ends_b, int32_t* blocks, int32_t* status,
                       void* workspace, size_t workspace_bytes, void* stream) {
    if (X < 1 || Y < 1 || nnz < 0 || n_moves < 0 || (long long)nnz > (long long)X * Y) return PBS_ERR_BAD_SHAPE;
    if ((long long)X * Y > (1ll << 30)) return PBS_ERR_TOO_LARGE;
    if (!row_start_ends_a || !col_start_ends_b || !status || (n_moves > 0 && !moves)) return PBS_ERR_NULL_POINTER;
    if (nnz > 0 && (!old_blocks || !cols_a || !rows_b || !blocks)) return PBS_ERR_NULL_POINTER;
    const size_t need = replace_ws_bytes(X, Y, nnz);
    if (need > 0 && (!workspace || workspace_bytes < need || !aligned16(workspace))) return PBS_ERR_WORKSPACE;
    return launch(replace_blocks_kernel, dim3(1), dim3(INDEX_THREADS), 0, static_cast<hipStream_t>(stream), old_blocks, moves, n_moves, X,
                  Y, nnz, cols_a, row_start_ends_a, rows_b, col_start_ends_b, blocks, status, static_cast<int*>(workspace));
}

size_t pbs_validate_indices_workspace_bytes(int nnz) { return nnz < 0 ? 0 : validate_ws_bytes(nnz); }

int pbs_validate_indices(const int32_t* cols_a, const int32_t* row_start_ends_a, const int32_t* rows_b,
                         const int32_t* col_start_ends_b, const int32_t* blocks, int X, int Y, int nnz, int32_t* status,
                         void* workspace, size_t workspace_bytes, void* stream) {
    if (X < 1 || Y < 1 || nnz < 0) return PBS_ERR_BAD_SHAPE;
    if ((long long)X * Y > (1ll << 30)) return PBS_ERR_TOO_LARGE;
    if (!row_start_ends_a || !col_start_ends_b || !status || (nnz > 0 && (!cols_a || !rows_b || !blocks))) return PBS_ERR_NULL_POINTER;
    const size_t need = validate_ws_bytes(nnz);
    if (need > 0 && (!workspace || workspace_bytes < need || !aligned16(workspace))) return PBS_ERR_WORKSPACE;
    return launch(validate_indices_kernel, dim3(1), dim3(INDEX_THREADS), 0, static_cast<hipStream_t>(stream), cols_a, row_start_ends_a,
                  rows_b, col_start_ends_b, blocks, X, Y, nnz, status, static_cast<int*>(workspace));
}

size_t pbs_blocksparse_matmul_plan_bytes(int n, int k) {
    if (n <= 0 || k <= 0 || (n % 32) || (k % 32)) return 0;
    return all_plan_bytes(n, k);
}

size_t pbs_blocksparse_matmul_plan_part_bytes(int n, int k) {
    if (n <= 0 || k <= 0 || (n % 32) || (k % 32)) return 0;
    return part_plan_bytes(n, k);
}

static int plan_checks(const int32_t* ptr, const int32_t* indices, int n, int k, int nnz, const void* plan, size_t plan_bytes) {
    if (n <= 0 || k <= 0 || nnz < 0 || (n % 32) || (k % 32)) return PBS_ERR_BAD_SHAPE;
    if ((long long)nnz > (long long)(n / 32) * (k / 32) || k > (1 << 24)) return PBS_ERR_TOO_LARGE;
    if (!ptr || !plan || (nnz > 0 && !indices)) return PBS_ERR_NULL_POINTER;
    if (!aligned16(plan) || plan_bytes < part_plan_bytes(n, k)) return PBS_ERR_WORKSPACE;
    return PBS_OK;
}

int pbs_blocksparse_matmul_plan_part(const int32_t* ptr, const int32_t* indices, int n, int k, int nnz, int part, void* plan,
                                     size_t plan_bytes, void* stream) {
    if (int rc = plan_checks(ptr, indices, n, k, nnz, plan, plan_bytes)) return rc;
    hipStream_t s = static_cast<hipStream_t>(stream);
    unsigned char* base = static_cast<unsigned char*>(plan);
    if (part & PART_LIST) {
        const ListArgs a{ptr, indices, n / 32, k / 32, nnz, reinterpret_cast<int*>(base)};
        if (int rc = launch(list_plan_kernel, dim3(list_plan_grid(n / 32)), dim3(256), 0, s, a)) return rc;
    }
    if ((part & PART_WIDE) && wide_plan_bytes(n, k)) {
        const int groups16 = (n / 32 + D16_NB - 1) / D16_NB;
        int* wide = reinterpret_cast<int*>(base + list_area_bytes(n, k));
        if (int rc = launch(dds16_plan_kernel, dim3(groups16), dim3(256), 0, s, ptr, indices, n / 32, k / 32, nnz, wide,
                            (int)dds16_plan_group_ints(k / 32), wide + (size_t)groups16 * dds16_plan_group_ints(k / 32))) return rc;
    }
    if ((part & PART_COLUMN) && column_plan_bytes(n, k)) {
        const int groups = column_groups(n);
        const int group_ints = (int)ddsc_plan_group_ints(k / 32);
        int* cols = reinterpret_cast<int*>(base + column_plan_offset(n, k));
        int* lists = reinterpret_cast<int*>(base + column_plan_offset(n, k) + column_table_bytes(n));
        if (int rc = launch(ddsc_cols_kernel, dim3(1), dim3(256), 0, s, ptr, n / 32, groups, nnz, cols)) return rc;
        if (int rc = launch(ddsc_plan_kernel, dim3(groups), dim3(256), 0, s, ptr, indices, cols, n / 32, k / 32, nnz, lists,
                            group_ints, lists + (size_t)groups * group_ints)) return rc;
        if (int rc = launch(ddsc_plan_ahead_kernel, dim3(groups), dim3(64), 0, s, k / 32, lists, group_ints)) return rc;
    }
    return PBS_OK;
}

int pbs_blocksparse_matmul_plan(const int32_t* ptr, const int32_t* indices, int n, int k, int nnz, void* plan,
                                size_t plan_bytes, void* stream) {
    if (int rc = plan_checks(ptr, indices, n, k, nnz, plan, plan_bytes)) return rc;
    if (plan_bytes < all_plan_bytes(n, k)) return PBS_ERR_WORKSPACE;
    if (int rc = pbs_blocksparse_matmul_plan_part(ptr, indices, n, k, nnz, PART_LIST | PART_WIDE | PART_COLUMN, plan, plan_bytes, stream))
        return rc;
    SlotTables t;
    for (int wi = 0; wi < PLAN_NWIDTHS; ++wi) {
        t.table[wi] = reinterpret_cast<int*>(static_cast<unsigned char*>(plan) + slot_table_offset(n, k, wi));
        t.groups[wi] = (int)width_groups(n, wi);
    }
    const int places = t.groups[PLAN_NWIDTHS - 1] * PLAN_PLACES;
    return launch(slot_tables_kernel, dim3((unsigned)(places < 16384 ? (places + 255) / 256 : 64)), dim3(256), 0,
                  static_cast<hipStream_t>(stream), t, n / 32);
}

int pbs_blocksparse_matmul_part(int64_t tokens, int n, int k, int nnz, int transpose, int dtype, int with_workspace) {
    if ((dtype != PBS_DTYPE_F32 && dtype != PBS_DTYPE_BF16) || tokens <= 0 || n <= 0 || k <= 0 || nnz < 0 || (n % 32) || (k % 32))
        return PART_LIST;
    return choose_product(dtype == PBS_DTYPE_F32 ? 4 : 2, tokens, n, k, nnz, transpose, with_workspace != 0).part;
}

size_t pbs_blocksparse_matmul_workspace_bytes(int64_t tokens, int n, int k, int nnz, int transpose, int dtype) {
    if (dtype != PBS_DTYPE_BF16 || !transpose || tokens <= 0 || n <= 0 || k <= 0 || nnz <= 0 || (n % 32) || (k % 32)) return 0;
    if ((long long)nnz > (long long)(n / 32) * (k / 32)) return 0;
    return choose_product(2, tokens, n, k, nnz, 1, true).part == PART_COLUMN ? (size_t)nnz * 2048 : 0;
}

size_t pbs_blocksparse_matmul_parts_bytes(int64_t tokens, int n, int k, int nnz, int transpose, int dtype) {
    if (dtype != PBS_DTYPE_F32 || tokens <= 0 || n <= 0 || k <= 0 || nnz <= 0 || (n % 32) || (k % 32)) return 0;
    if ((long long)nnz > (long long)(n / 32) * (k / 32)) return 0;
    return split_kernel_fits(tokens, n, k, nnz) ? split_workspace_bytes(nnz) : 0;
}

int pbs_blocksparse_matmul(const void* dense_a, const void* data, const void* plan, const void* bias, void* dense_out,
                           int64_t tokens, int n, int k, int nnz, int transpose, int dtype, void* stream) {
    return pbs_blocksparse_matmul_ws(dense_a, data, plan, bias, dense_out, tokens, n, k, nnz, transpose, dtype, nullptr, 0,
                                     stream);
}

static int matmul_checks(const void* dense_a, const void* data, const void* plan, const void* dense_out, int64_t tokens, int n, int k, int nnz, int dtype) {
    if (dtype != PBS_DTYPE_F32 && dtype != PBS_DTYPE_BF16) return PBS_ERR_BAD_DTYPE;
    if (tokens < 0 || n <= 0 || k <= 0 || nnz < 0 || (n % 32) || (k % 32)) return PBS_ERR_BAD_SHAPE;
    if (tokens > (1ll << 30) || (long long)nnz > (long long)(n / 32) * (k / 32) || k > (1 << 24)) return PBS_ERR_TOO_LARGE;
    if (tokens == 0) return PBS_OK;
    if (!dense_a || !plan || !dense_out) return PBS_ERR_NULL_POINTER;
    if (nnz > 0 && !data) return PBS_ERR_NULL_POINTER;
    if (!aligned16(dense_a) || !aligned16(data) || !aligned16(dense_out) || !aligned16(plan)) return PBS_ERR_MISALIGNED;
    return PBS_OK;
}

int pbs_blocksparse_matmul_ws(const void* dense_a, const void* data, const void* plan, const void* bias, void* dense_out,
                              int64_t tokens, int n, int k, int nnz, int transpose, int dtype, void* workspace,
                              size_t workspace_bytes, void* stream) {
    if (int rc = matmul_checks(dense_a, data, plan, dense_out, tokens, n, k, nnz, dtype)) return rc;
    if (tokens == 0) return PBS_OK;
    DdsArgs g;
    g.a = dense_a;
    g.data = data;
    g.plan = static_cast<const int*>(plan);
    g.bias = bias;
    g.out = dense_out;
    g.M = (int)tokens;
    g.N = n;
    g.K = k;
    g.nnz = nnz;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == PBS_DTYPE_F32) {
        return transpose ? dispatch_dds<float, 0>(g, workspace, workspace_bytes, s) : dispatch_dds<float, 1>(g, workspace, workspace_bytes, s);
    }
    return transpose ? dispatch_dds<bf16_t, 0>(g, workspace, workspace_bytes, s)
                     : dispatch_dds<bf16_t, 1>(g, nullptr, 0, s);
}

static bool back_sizes_ok(int64_t tokens, int out_features, int in_features, int nnz, int dtype) {
    return tokens > 0 && out_features > 0 && in_features > 0 && nnz >= 0 && out_features % 32 == 0 && in_features % 32 == 0 &&
           (dtype == PBS_DTYPE_F32 || dtype == PBS_DTYPE_BF16);
}

size_t pbs_blocksparse_matmul_back_units_bytes(int64_t tokens, int out_features, int in_features, int nnz, int dtype) {
    if (!back_sizes_ok(tokens, out_features, in_features, nnz, dtype)) return 0;
    return plan_back(dtype, tokens, out_features, in_features, nnz, false, true).slices > 0 ? unit_table_bytes(out_features, nnz, unit_lists_only(out_features / 32)) : 0;
}

int pbs_blocksparse_matmul_back_units(const int32_t* row_start_ends_a, const int32_t* cols_a, int out_features, int in_features,
                                      int nnz, void* units, size_t units_bytes, void* stream) {
    if (out_features <= 0 || in_features <= 0 || nnz < 0 || (out_features % 32) || (in_features % 32)) return PBS_ERR_BAD_SHAPE;
    if ((long long)nnz > (long long)(out_features / 32) * (in_features / 32)) return PBS_ERR_TOO_LARGE;
    if (!row_start_ends_a || (nnz > 0 && !cols_a) || !units) return PBS_ERR_NULL_POINTER;
    if (!aligned16(units)) return PBS_ERR_MISALIGNED;
    const int only = unit_lists_only(out_features / 32);
    if (units_bytes < unit_table_bytes(out_features, nnz, only)) return PBS_ERR_WORKSPACE;
    return build_units(row_start_ends_a, cols_a, out_features, in_features, nnz, only, units, static_cast<hipStream_t>(stream));
}

size_t pbs_blocksparse_matmul_back_bias_workspace_bytes(int64_t tokens, int out_features, int in_features, int nnz, int dtype) {
    if (!back_sizes_ok(tokens, out_features, in_features, nnz, dtype)) return 0;
    return plan_back(dtype, tokens, out_features, in_features, nnz, true, true).partial_bytes;
}

size_t pbs_blocksparse_matmul_back_workspace_bytes(int64_t tokens, int out_features, int in_features, int nnz,
                                                   int dtype) {
    if (!back_sizes_ok(tokens, out_features, in_features, nnz, dtype) || nnz == 0) return 0;
    const BackPlan p = plan_back(dtype, tokens, out_features, in_features, nnz, false, false);
    return p.partial_bytes + (p.slices > 0 ? unit_table_bytes(out_features, nnz, p.per_unit) : 0);
}

int pbs_blocksparse_derive(const int32_t* row_start_ends_a, const int32_t* cols_a, const int32_t* col_start_ends_b, const int32_t* rows_b,
                           int out_features, int in_features, int nnz, void* plan_forward, size_t plan_forward_bytes, void* plan_input,
                           size_t plan_input_bytes, void* units, size_t units_bytes, void* stream) {
    if (int rc = plan_checks(row_start_ends_a, cols_a, out_features, in_features, nnz, plan_forward, plan_forward_bytes)) return rc;
    if (int rc = plan_checks(col_start_ends_b, rows_b, in_features, out_features, nnz, plan_input, plan_input_bytes)) return rc;
    if (units && !aligned16(units)) return PBS_ERR_MISALIGNED;
    if (units && units_bytes < unit_table_bytes(out_features, nnz, unit_lists_only(out_features / 32))) return PBS_ERR_WORKSPACE;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int N = out_features / 32, K = in_features / 32;
    const bool with_units = units && !unit_prefix_bytes(out_features);   // (very tall matrices need a launch before that one)
    DeriveArgs a;
    a.list[0] = ListArgs{row_start_ends_a, cols_a, N, K, nnz, static_cast<int*>(plan_forward)};
    a.list[1] = ListArgs{col_start_ends_b, rows_b, K, N, nnz, static_cast<int*>(plan_input)};
    a.grid[0] = (int)list_plan_grid(N);
    a.grid[1] = (int)list_plan_grid(K);
    a.units = UnitArgs{row_start_ends_a, cols_a, nnz, N, K, nullptr, 0, with_units ? static_cast<int*>(units) : nullptr};
    const long long grid = (long long)a.grid[0] + a.grid[1] + (with_units ? unit_table_grid(N, nnz, 0) : 0);
    if (int rc = launch(derive_kernel, dim3((unsigned)grid), dim3(256), 0, s, a)) return rc;
    return units && !with_units ? build_units(row_start_ends_a, cols_a, out_features, in_features, nnz, unit_lists_only(N), units, s) : PBS_OK;
}

static int back_checks(const BackArgs& a, int64_t tokens, int dtype) {
    if (dtype != PBS_DTYPE_F32 && dtype != PBS_DTYPE_BF16) return PBS_ERR_BAD_DTYPE;
    if (tokens < 0 || a.N <= 0 || a.K <= 0 || a.nnz < 0 || (a.N % 32) || (a.K % 32)) return PBS_ERR_BAD_SHAPE;
    if (tokens > (1ll << 30) || (long long)a.nnz > (long long)(a.N / 32) * (a.K / 32)) return PBS_ERR_TOO_LARGE;
    if (a.nnz == 0 && !a.bias_out) return PBS_OK;
    if (!a.ptr || (a.nnz > 0 && (!a.idx || !a.out))) return PBS_ERR_NULL_POINTER;
    if (tokens > 0 && (!a.g || !a.x)) return PBS_ERR_NULL_POINTER;
    if (!aligned16(a.g) || !aligned16(a.x) || !aligned16(a.out) || !aligned16(a.bias_out) || !aligned16(a.units)) return PBS_ERR_MISALIGNED;
    return PBS_OK;
}
static int back(const BackArgs& a, int64_t tokens, int dtype, void* workspace, size_t workspace_bytes, void* stream,
                size_t workspace_limit = ROW_WORKSPACE_BYTES) {
    if (int rc = back_checks(a, tokens, dtype)) return rc;
    if (a.nnz == 0 && !a.bias_out) return PBS_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (tokens == 0) {
        const size_t esz = dtype == PBS_DTYPE_F32 ? 4 : 2;
        auto zero = [&](void* p, size_t values) {
            const size_t nwords = values * esz / 4;
            return launch(fill_zero_kernel, dim3((unsigned)((nwords + 255) / 256)), dim3(256), 0, s, static_cast<uint32_t*>(p), nwords);
        };
        if (a.nnz > 0)
            if (int rc = zero(a.out, (size_t)a.nnz * 1024)) return rc;
        return a.bias_out ? zero(a.bias_out, a.N) : PBS_OK;
    }
    const BackPlan p = plan_back(dtype, tokens, a.N, a.K, a.nnz, a.bias_out != nullptr, a.lists, workspace_limit);
    if (p.slices == 0) return a.bias_out ? launch_rectangles<true>(a, p, workspace, workspace_bytes, s) : launch_rectangles<false>(a, p, workspace, workspace_bytes, s);
    return dtype == PBS_DTYPE_F32 ? launch_row<float>(a, p, workspace, workspace_bytes, s) : launch_row<bf16_t>(a, p, workspace, workspace_bytes, s);
}

int pbs_blocksparse_matmul_back(const void* dense_a, const void* dense_b, const int32_t* row_start_ends_a,
                                const int32_t* cols_a, void* data_out, int64_t tokens, int out_features,
                                int in_features, int nnz, int dtype, void* workspace, size_t workspace_bytes,
                                void* stream) {
    const BackArgs a{dense_a, dense_b, row_start_ends_a, cols_a, nullptr, false, data_out, nullptr, (int)tokens, out_features, in_features, nnz, nullptr, nullptr};
    return back(a, tokens, dtype, workspace, workspace_bytes, stream);
}

int pbs_blocksparse_matmul_back_bias(const void* dense_a, const void* dense_b, const int32_t* row_start_ends_a,
                                     const int32_t* cols_a, const void* units, void* data_out, void* bias_out, int64_t tokens,
                                     int out_features, int in_features, int nnz, int dtype, void* workspace, size_t workspace_bytes,
                                     void* stream) {
    if (!units && pbs_blocksparse_matmul_back_units_bytes(tokens, out_features, in_features, nnz, dtype) > 0) return PBS_ERR_NULL_POINTER;
    const BackArgs a{dense_a, dense_b, row_start_ends_a, cols_a, units, true, data_out, bias_out, (int)tokens, out_features, in_features, nnz, nullptr, nullptr};
    return back(a, tokens, dtype, workspace, workspace_bytes, stream);
}

// A workspace of both products: the slices of the weight gradient, and behind them the blocks in parts.
static size_t slices_bytes(int64_t tokens, int out_features, int in_features, int nnz, int dtype) {
    return (pbs_blocksparse_matmul_back_bias_workspace_bytes(tokens, out_features, in_features, nnz, dtype) + 255) / 256 * 256;
}
size_t pbs_blocksparse_linear_back_workspace_bytes(int64_t tokens, int out_features, int in_features, int nnz, int dtype) {
    return slices_bytes(tokens, out_features, in_features, nnz, dtype) +
           pbs_blocksparse_matmul_parts_bytes(tokens, in_features, out_features, nnz, 0, dtype);
}

int pbs_blocksparse_linear_back(const void* grad_output, const void* input, const void* data, const void* plan_input, const int32_t* row_start_ends_a,
                                const int32_t* cols_a, const void* units, void* grad_input, void* data_out, void* bias_out, int64_t tokens,
                                int out_features, int in_features, int nnz, int dtype, void* workspace, size_t workspace_bytes, void* stream) {
    if (int rc = matmul_checks(grad_output, data, plan_input, grad_input, tokens, in_features, out_features, nnz, dtype)) return rc;
    const size_t slices = slices_bytes(tokens, out_features, in_features, nnz, dtype),
                 parts = pbs_blocksparse_matmul_parts_bytes(tokens, in_features, out_features, nnz, 0, dtype);
    if (slices + parts > 0 && (!workspace || workspace_bytes < slices + parts || !aligned16(workspace))) return PBS_ERR_WORKSPACE;
    if (!units && pbs_blocksparse_matmul_back_units_bytes(tokens, out_features, in_features, nnz, dtype) > 0) return PBS_ERR_NULL_POINTER;
    void* const behind = parts ? static_cast<unsigned char*>(workspace) + slices : nullptr;
    const DdsArgs g{grad_output, data, static_cast<const int*>(plan_input), nullptr, grad_input, (int)tokens, in_features, out_features, nnz};
    BackArgs a{grad_output, input, row_start_ends_a, cols_a, units, true, data_out, bias_out, (int)tokens, out_features, in_features, nnz, nullptr, nullptr};
    if (int rc = back_checks(a, tokens, dtype)) return rc;   // (before the input gradient is launched)
    auto input_gradient = [&](bool parts_ready) {
        if (tokens == 0) return (int)PBS_OK;
        hipStream_t s = static_cast<hipStream_t>(stream);
        return dtype == PBS_DTYPE_F32 ? dispatch_dds<float, 1>(g, behind, parts, s, parts_ready) : dispatch_dds<bf16_t, 1>(g, nullptr, 0, s);
    };
    // with a launch that adds the slices, the blocks are split by that one too, and the input gradient comes last
    const bool together = parts > 0 && plan_back(dtype, tokens, out_features, in_features, nnz, bias_out != nullptr, true).partials > 0;
    if (together) {
        a.data = data;
        a.parts = behind;
        if (int rc = back(a, tokens, dtype, workspace, slices, stream)) return rc;
        return input_gradient(true);
    }
    if (int rc = input_gradient(false)) return rc;
    return back(a, tokens, dtype, workspace, slices, stream);
}

// ---- the reference's own signature of the sparse-output product ----
struct BackBlocksLayout {
    size_t row_ptr, cols_a, owner, a_t, b_t, inner, total;   // byte offsets into the workspace; inner = the split workspace
};
static inline size_t round256(size_t v) { return (v + 255) / 256 * 256; }
static BackBlocksLayout back_blocks_layout(int64_t tokens, int out_features, int in_features, int nnz, int dtype,
                                           int a_row_major, int b_row_major) {
    BackBlocksLayout l;
    const size_t X = out_features / 32, Y = in_features / 32, esz = dtype == PBS_DTYPE_F32 ? 4 : 2;
    size_t off = 0;
    l.row_ptr = off;
    off += round256((X + 1) * sizeof(int32_t));
    l.cols_a = off;
    off += round256((size_t)nnz * 2 * sizeof(int32_t));
    l.owner = off;
    off += round256(X * Y * sizeof(int));
    l.a_t = off;
    if (!a_row_major) off += round256((size_t)tokens * out_features * esz);
    l.b_t = off;
    if (!b_row_major) off += round256((size_t)tokens * in_features * esz);
    l.inner = off;
    off += round256(pbs_blocksparse_matmul_back_workspace_bytes(tokens, out_features, in_features, nnz, dtype));
    l.total = off;
    return l;
}

size_t pbs_blocksparse_matmul_back_blocks_workspace_bytes(int64_t tokens, int out_features, int in_features, int nnz,
                                                          int dtype, int a_row_major, int b_row_major) {
    if (tokens < 0 || out_features <= 0 || in_features <= 0 || nnz <= 0) return 0;
    if ((out_features % 32) || (in_features % 32)) return 0;
    if (dtype != PBS_DTYPE_F32 && dtype != PBS_DTYPE_BF16) return 0;
    return back_blocks_layout(tokens, out_features, in_features, nnz, dtype, a_row_major, b_row_major).total;
}

int pbs_blocksparse_matmul_back_blocks(const void* dense_a, int a_row_major, const void* dense_b, int b_row_major,
                                       void* data_out, int64_t tokens, int out_features, int in_features,
                                       const int32_t* blocks, int nnz, int dtype, void* workspace, size_t workspace_bytes,
                                       void* stream) {
    if (dtype != PBS_DTYPE_F32 && dtype != PBS_DTYPE_BF16) return PBS_ERR_BAD_DTYPE;
    if (tokens < 0 || out_features <= 0 || in_features <= 0 || nnz < 0 || (out_features % 32) || (in_features % 32))
        return PBS_ERR_BAD_SHAPE;
    if (tokens > (1ll << 30) || (long long)nnz > (long long)(out_features / 32) * (in_features / 32))
        return PBS_ERR_TOO_LARGE;
    if (nnz == 0) return PBS_OK;
    if (!blocks || !data_out) return PBS_ERR_NULL_POINTER;
    if (tokens > 0 && (!dense_a || !dense_b)) return PBS_ERR_NULL_POINTER;
    if (!aligned16(dense_a) || !aligned16(dense_b) || !aligned16(data_out)) return PBS_ERR_MISALIGNED;
    const BackBlocksLayout l = back_blocks_layout(tokens, out_features, in_features, nnz, dtype, a_row_major, b_row_major);
    if (!workspace || workspace_bytes < l.total || !aligned16(workspace)) return PBS_ERR_WORKSPACE;
    unsigned char* ws = static_cast<unsigned char*>(workspace);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int X = out_features / 32, Y = in_features / 32;
    int32_t* row_ptr = reinterpret_cast<int32_t*>(ws + l.row_ptr);
    int32_t* cols_a = reinterpret_cast<int32_t*>(ws + l.cols_a);
    int* owner = reinterpret_cast<int*>(ws + l.owner);
    const long long positions = (long long)X * Y;
    if (int rc = launch(blocks_owner_clear_kernel, dim3((unsigned)((positions + 255) / 256)), dim3(256), 0, s, owner, positions)) return rc;
    if (int rc = launch(blocks_owner_kernel, dim3((unsigned)((nnz + 255) / 256)), dim3(256), 0, s, blocks, nnz, X, Y, owner)) return rc;
    if (int rc = launch(csr_from_owner_kernel, dim3(1), dim3(INDEX_THREADS), 0, s, owner, X, Y, cols_a, row_ptr)) return rc;
    // an operand given with the tokens along its rows' direction ([features, tokens]) is brought to [tokens, features]
    auto to_row_major = [&](const void* src, size_t off, int features) -> int {
        const dim3 grid((unsigned)((tokens + 31) / 32), (unsigned)((features + 31) / 32));
        if (dtype == PBS_DTYPE_F32)
            return launch(transpose_dense_kernel<uint32_t>, grid, dim3(256), 0, s, static_cast<const uint32_t*>(src),
                          reinterpret_cast<uint32_t*>(ws + off), (long long)features, (long long)tokens);
        return launch(transpose_dense_kernel<uint16_t>, grid, dim3(256), 0, s, static_cast<const uint16_t*>(src),
                      reinterpret_cast<uint16_t*>(ws + off), (long long)features, (long long)tokens);
    };
    const void* a = dense_a;
    const void* b = dense_b;
    if (!a_row_major && tokens > 0) {
        if (int rc = to_row_major(dense_a, l.a_t, out_features)) return rc;
        a = ws + l.a_t;
    }
    if (!b_row_major && tokens > 0) {
        if (int rc = to_row_major(dense_b, l.b_t, in_features)) return rc;
        b = ws + l.b_t;
    }
    return pbs_blocksparse_matmul_back(a, b, row_ptr, cols_a, data_out, tokens, out_features, in_features, nnz, dtype,
                                       ws + l.inner, l.total - l.inner, stream);
}

size_t pbs_blocksparse_matmul_back_noalloc_max_bytes(void) { return PBS_NOALLOC_SCRATCH_BYTES; }

int pbs_blocksparse_matmul_back_noalloc_init(void) {
    void* ws = nullptr;
    return scratch_of_current_device(&ws);
}

int pbs_blocksparse_matmul_back_noalloc(const void* dense_a, const void* dense_b, const int32_t* row_start_ends_a,
                                        const int32_t* cols_a, void* data_out, int64_t tokens, int out_features,
                                        int in_features, int nnz, int dtype, void* stream) {
    // the array limits the number of slices of the row kernel; the rectangles' is fixed
    const BackArgs a{dense_a, dense_b, row_start_ends_a, cols_a, nullptr, false, data_out, nullptr, (int)tokens, out_features, in_features, nnz, nullptr, nullptr};
    size_t need = 0, limit = 0;
    if (back_sizes_ok(tokens, out_features, in_features, nnz, dtype) && nnz > 0) {
        const size_t table = unit_table_bytes(out_features, nnz, ROW_NB);
        limit = (size_t)PBS_NOALLOC_SCRATCH_BYTES > table ? (size_t)PBS_NOALLOC_SCRATCH_BYTES - table : 0;
        const BackPlan p = plan_back(dtype, tokens, out_features, in_features, nnz, false, false, limit);
        need = p.partial_bytes + (p.slices > 0 ? unit_table_bytes(out_features, nnz, p.per_unit) : 0);
    }
    if (need > (size_t)PBS_NOALLOC_SCRATCH_BYTES) return PBS_ERR_SCRATCH;
    void* ws = nullptr;
    if (need > 0) {
        if (int rc = scratch_of_current_device(&ws)) return rc;
    }
    return back(a, tokens, dtype, ws, need, stream, limit);
}

int pbs_protocol_failures(unsigned* count) {
    if (!count) return PBS_ERR_NULL_POINTER;
    return (int)hipMemcpyFromSymbol(count, HIP_SYMBOL(g_protocol_failures), sizeof(unsigned), 0, hipMemcpyDeviceToHost);
}

const char* pbs_blocksparse_matmul_kernel_name(int64_t tokens, int n, int k, int nnz, int transpose, int dtype,
                                               int with_workspace) {
    if ((dtype != PBS_DTYPE_F32 && dtype != PBS_DTYPE_BF16) || tokens <= 0 || n <= 0 || k <= 0 || (n % 32) || (k % 32)) return "";
    const ProductChoice c = choose_product(dtype == PBS_DTYPE_F32 ? 4 : 2, tokens, n, k, nnz, transpose, with_workspace != 0);
    if (dtype == PBS_DTYPE_F32 && with_workspace && nnz > 0 && split_kernel_fits(tokens, n, k, nnz)) return "split_kernel";
    if (dtype == PBS_DTYPE_F32 && choose_walk(tokens, n, k, nnz)) return "walk_kernel";
    return c.part == PART_COLUMN ? "ddsc_kernel" : (c.part == PART_WIDE ? "dds16_kernel" : (!c.panel.splits ? "stream_kernel" : (c.panel.ways ? "panel_chunk_kernel" : "panel_kernel")));
}

const char* pbs_blocksparse_matmul_kernel_form(int64_t tokens, int n, int k, int nnz, int transpose, int dtype, int with_workspace) {
    static thread_local char text[96];
    const char* name = pbs_blocksparse_matmul_kernel_name(tokens, n, k, nnz, transpose, dtype, with_workspace);
    std::snprintf(text, sizeof text, "%s%s", name, !std::strcmp(name, "ddsc_kernel") && touches(tokens, n, k, nnz) ? ", lines ahead" : "");
    return text;
}

const char* pbs_blocksparse_matmul_back_kernel_name(int64_t tokens, int out_features, int in_features, int nnz, int dtype) {
    if ((dtype != PBS_DTYPE_F32 && dtype != PBS_DTYPE_BF16) || tokens <= 0 || out_features <= 0 || in_features <= 0 ||
        nnz <= 0 || (out_features % 32) || (in_features % 32))
        return "";
    const BackPlan p = plan_back(dtype, tokens, out_features, in_features, nnz, false, true);
    if (p.slices > 0 && p.split) return p.slices > 1 ? "sdd_split_kernel + sdd_reduce_kernel" : "sdd_split_kernel";
    if (p.slices > 0) return p.slices > 1 ? "sdd_row_kernel + sdd_reduce_kernel" : "sdd_row_kernel";
    return p.rect.nsplit > 1 ? "sdd_bf16_kernel + sdd_reduce_kernel" : "sdd_bf16_kernel";
}

const char* pbs_blocksparse_matmul_back_kernel_form(int64_t tokens, int out_features, int in_features, int nnz, int dtype) {
    static thread_local char text[128];
    const char* name = pbs_blocksparse_matmul_back_kernel_name(tokens, out_features, in_features, nnz, dtype);
    if (!name[0] || plan_back(dtype, tokens, out_features, in_features, nnz, false, true).slices > 0) return name;
    const SddPlan p = plan_back(dtype, tokens, out_features, in_features, nnz, false, true).rect;
    std::snprintf(text, sizeof text, "%s, %d %sbands of %d rows x %d rectangles x %d slices", name, p.tiles_r, p.even ? "even " : "", p.rows, p.tiles_c, p.nsplit);
    return text;
}

}  // extern "C"
