// dense x block-sparse -> dense in fp32 on the bf16 matrix cores (forward and input gradient of larger problems).
//
// The fp32 matrix instruction multiplies at a sixteenth of the bf16 rate.  A float is the sum of three bfloat16 values without a rest
// (24 bits of significand in three times 8), so a product of two floats is nine products of bfloat16 values.  The three smallest, each
// below 2^-25 of the whole and together at most 2^-24 of it, are left out: six bf16 instructions do the work of an fp32 instruction that takes
// 16 times as long (G. Henry, P. T. P. Tang, A. Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for higher-precision
// computations", ARITH 2019).
//
// Sums are float32.  A block's twelve products (two halves of k) are summed by themselves, the small ones first, and join the column's total with
// one rounding per block.  The matrix instruction cuts what is far below its largest term off, towards minus infinity (a mean error of -3e-8 of the
// results' size at 48 blocks), so every other k-block is multiplied with the dense operand's sign changed and subtracted (mean error below 1e-9).
// Distance from float64 in units of 1e-7, in the chains of fp32 instructions of stream_kernel, in one chain over the column here, and as it is:
//   768 -> 3072 density 0.5   2.6  1.1  0.8      3072 -> 768 density 0.5   3.6  2.3  1.4      4096 -> 4096 density 0.25   2.9  1.9  1.1
//   the same layers with operands between 0 and 1   1.5  1.1  0.6      1.5  2.1  1.1      1.3  1.7  0.9
// and of products of a single value, which no sum averages, 0.25 and 0.35 (at most 0.6 and 1.6).
// The sums by block cost 1 to 4 % of a product against the one chain (32 vector instructions per block and wave, in a kernel bound by power); blocks in
// pairs would cost half of that, but leave the mean error: a pair has no sign of its own in panels that eight columns share.
//
// Range.  Operands are scaled by 2^30 when they are split, so that the third part of the smallest normal float is still a
// normal bfloat16; the result is scaled back.  Whatever does not fit (an operand above 2^97, a result above 2^67, infinities and
// NaN) leaves a result that is not finite, and such results alone are computed again with fp32 instructions, in the epilogue.
//
// What bounds the work.  Splitting costs 6.5 vector instructions per value, 1.3 times what the matrix instructions of a 64 x 32 tile
// take if every wave splits what it multiplies (vector and matrix instructions of different waves overlap, apart from
// about 8 cycles that each matrix instruction holds up the issue of the others).  So a value is split once for
// many users: the blocks by a launch of their own (split_blocks_kernel, into a workspace, in the order the fragments are loaded in), the
// dense operand once per 8 block columns, by waves that do nothing else.  What is left is mostly power: the matrix cores are busy 0.52 to 0.56 of
// the time at 1.56 GHz (with zeros for operands the same cycles pass at 2.0 GHz).
// us, stream_kernel -> here (with the launch that splits the blocks): 768 -> 3072 density 0.5, 4096 tokens 92 -> 65, 3072 -> 768 83 -> 66, 768 -> 768
// density 0.5, 16384 tokens 92 -> 64, 4096 -> 4096 density 0.25, 16384 tokens 1216 -> 870.
//
// A workgroup takes 64 tokens x 8 block columns at a time.  Waves 0-7 multiply, one block column each: per block, 6 KB of fragments from
// memory (asked for an item ahead) and 12 KB from the panel ring in LDS for 24 instructions of 32 cycles.  Waves 8-11 load the panel of a k-block
// (64 tokens x 32 features), split it and write it to the ring (12 slots of 12 KB).  Progress words in LDS instead of barriers, so that columns with
// fewer blocks in a stretch of k run ahead and SIMDs do not wait for each other:
//   landed[s]   ring slot s holds step landed[s] - 1 (written by the wave that filled it, when its writes are done)
//   done[w]     the step wave w still needs: it has read every earlier one
// Every wait polls with s_sleep and is bounded; one that runs into its bound makes the results NaN and is counted.
// Workgroups are persistent, one per CU: units (token tile, group of columns) are dealt so that an XCD's workgroups share panels
// and blocks in its L2.  Columns are ranked by their number of blocks in the list plan (pbs_stream.h) and dealt to the groups and SIMDs in turn.
// A wave goes through its column by k-block whatever the tile, so a token's result has the same bits in any call that this kernel serves.
// Measured and not kept: blocks of whole tiles two items ahead (waves with 32 tokens have the registers, below), or touched three items ahead for the L2 (7 % and more slower), wave priorities (2 to 6 %
// slower), another order of the six products (nothing), rings of 8 slots (3 % slower); columns of equal length to a group (a group waits for its longest
// column, but its units then differ: even patterns 3 % slower, uneven ones 0.74 to 1.16 times as fast); fewer columns in halves where their groups take
// another round of units (up to 1.38 times faster there, but short columns pay for the choice: 1 % slower on average, uneven patterns too).
#pragma once
#include "pbs_common.h"
#include "pbs_sdd.h"
#include "pbs_stream.h"

namespace pbs {

constexpr int SP_NC = 8;                 // multiplying waves = block columns of a group
constexpr int SP_NP = 4;                 // waves that fill the ring
constexpr int SP_MAX_UNITS = 64;         // of a workgroup: their heads are kept in LDS
constexpr int SP_SPIN_LIMIT = 1 << 20;
constexpr int SP_BLOCK_BYTES = 6144;     // a block's three parts
constexpr float SP_SCALE = 0x1p30f, SP_UNSCALE = 0x1p-60f;
constexpr int SP_BM = 64;                // tokens of a tile (of a low one 32)
constexpr int SP_MORE = 3;               // (with more groups than that more, as with that many)
constexpr int SP_RS = 12;                // ring slots; a multiple of SP_NP: a slot has one writer
constexpr int SP_PLANE = SP_BM * 64;     // one part of a panel: 64 bytes per token
constexpr int SP_SLOT = 3 * SP_PLANE;
constexpr int SP_LDS = SP_RS * SP_SLOT + SP_NC * SP_MAX_UNITS * 16 + 256;
static_assert(SP_RS % SP_NP == 0 && SP_LDS <= 160 * 1024, "a slot has one writer");

// two values into their three parts, packed in pairs
static __device__ __forceinline__ void split2(float a0, float a1, uint32_t& h, uint32_t& m, uint32_t& l) {
    // as a vector: one instruction, where two conversions and an or take four; and opaque, or every part is converted again to be taken off
    auto pack = [](float x, float y) __attribute__((always_inline)) {
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        uint32_t p = __builtin_bit_cast(uint32_t, bf16x2{static_cast<__bf16>(x), static_cast<__bf16>(y)});
        asm("" : "+v"(p));
        return p;
    };
    auto rest = [](float& x, float& y, uint32_t p) __attribute__((always_inline)) {   // exact
        x -= __uint_as_float(p << 16);
        y -= __uint_as_float(p & 0xffff0000u);
    };
    h = pack(a0, a1);
    rest(a0, a1, h);
    m = pack(a0, a1);
    rest(a0, a1, m);
    l = pack(a0, a1);
}

// The sign bit of the dense operand in a k-block: the parity of the ones in its number, so that any regular choice of k-blocks has as many of either
// kind.
static __device__ __forceinline__ int block_sign(int kb) { return (__popc((unsigned)kb) & 1) << 31; }
static __device__ __forceinline__ float with_sign(float v, int sign_uniform) {
    return __uint_as_float(__builtin_amdgcn_readfirstlane((int)__float_as_uint(v) ^ sign_uniform));
}

// The blocks in parts, as fragments: block b = [half q of k][part][lane = 32 h + n][8 k values], k = 16 q + 8 h + e, 6 KB.  One wave
// per block.  TRANS as in stream_kernel: 0: stored [k][n], 1: stored [n][k].
template <int TRANS>
static __device__ __forceinline__ void split_blocks(const float* __restrict__ data, unsigned char* __restrict__ parts, int nnz, int block) {
    const int lane = threadIdx.x & 63;
    const int b = block * 4 + (threadIdx.x >> 6);
    if (b >= nnz) return;
    const float* src = data + (size_t)b * 1024;
    unsigned char* dst = parts + (size_t)b * SP_BLOCK_BYTES + lane * 16;
    const int n = lane & 31, h = lane >> 5;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        float v[8];
        if constexpr (TRANS) {
            const float4 lo = *reinterpret_cast<const float4*>(src + n * 32 + 16 * q + 8 * h);
            const float4 hi = *reinterpret_cast<const float4*>(src + n * 32 + 16 * q + 8 * h + 4);
            v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
            v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = src[(16 * q + 8 * h + e) * 32 + n];
        }
        uint32_t p[3][4];
#pragma unroll
        for (int e = 0; e < 4; ++e) split2(v[2 * e] * SP_SCALE, v[2 * e + 1] * SP_SCALE, p[0][e], p[1][e], p[2][e]);
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<uint4*>(dst + (q * 3 + i) * 1024) = make_uint4(p[i][0], p[i][1], p[i][2], p[i][3]);
    }
}
static inline unsigned split_blocks_grid(int nnz) { return (unsigned)((nnz + 3) / 4); }
template <int TRANS>
__global__ __launch_bounds__(256) void split_blocks_kernel(const float* __restrict__ data, unsigned char* __restrict__ parts, int nnz) {
    split_blocks<TRANS>(data, parts, nnz, blockIdx.x);
}
// The sums of the slices of a weight gradient, and behind them the blocks of the input gradient that follows: behind a large kernel either takes 5.3 us
// as a launch of its own, whatever its size.  Training steps, us, with two launches and with this one: 3072 -> 768 density 0.25 in Zipf rows, 4096 tokens
// 164.1 and 155.5; 768 -> 768 density 0.5, 16384 tokens 229.3 and 224.7; 768 -> 3072 density 0.5, 4096 tokens 230.4 and 230.9 (the card's power: what the pause
// took, the kernel behind it took less).
__global__ __launch_bounds__(256) void sdd_reduce_split_kernel(const float* partial, float* out, size_t n, float* bias_out, size_t total, int nsplit,
                                                               unsigned reducing, const float* __restrict__ data, unsigned char* __restrict__ parts, int nnz) {
    if (blockIdx.x < reducing) sdd_reduce(partial, out, n, bias_out, total, nsplit, blockIdx.x);
    else split_blocks<1>(data, parts, nnz, (int)(blockIdx.x - reducing));
}

struct SplitArgs {
    const float* a;               // [M, K] row-major
    const float* data;            // [nnz*32, 32], as stored
    const unsigned char* parts;   // split_blocks_kernel
    const int* plan;              // the list plan
    const float* bias;            // nullptr or [N]
    float* out;                   // [M, N] row-major
    int M, N, K;
    int tiles[SP_MORE + 1];       // of 64 tokens, the others of 32 behind them; with so many groups more than without heavy columns
    int heavy;                    // columns of more blocks than this take two waves
    int tile_block;               // units are ordered by blocks of this many token tiles, then groups, then tiles
};

template <int TRANS>
__global__ __launch_bounds__((SP_NC + SP_NP) * 64, 3) void split_kernel(SplitArgs g) {
    constexpr int RS = SP_RS, SLOT = SP_SLOT, PLANE = SP_PLANE;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    int4* const s_heads = reinterpret_cast<int4*>(smem + RS * SLOT);                  // [SP_NC][SP_MAX_UNITS]
    int* const s_landed = reinterpret_cast<int*>(s_heads + SP_NC * SP_MAX_UNITS);   // [RS]
    int* const s_done = s_landed + RS;                            // [SP_NC]
    int* const s_fail = s_done + SP_NC;

    const int lane = lane_now();   // (what is kept of the thread's number over the multiplying waves' loops would be spilled)
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int KB = g.K >> 5, ncols = g.N >> 5;

    // A column of many more blocks than the others keeps its wave busy when all others are done.  So the columns of more than twice the average are
    // taken by two waves, 32 tokens of a tile each, in more groups if need be (3072 -> 768 with Zipf rows, 96 blocks of 24 on average, 4096 tokens: 66 -> 54 us
    // with the launch that splits the blocks).  Splitting more of them, or wherever a sum of rounds and longest stays says so, costs even patterns up to
    // 40 % (another group is another time that the panels are split).  Which tiles are full follows from the groups there are: with those of even columns,
    // 3072 -> 768 with Zipf rows, 8192 tokens took 129 us (98), 3360 -> 3488 density 0.32, 1688 tokens 158 (117), level where there are no heavy columns.
    // Place v of the dealing: below 2 * heavy half v % 2 of column v / 2 of the ranking, else column v - heavy.
    int heavy = 0;
    {
        const int2* ranked = reinterpret_cast<const int2*>(g.plan);
        bool more = true;
        for (int c0 = 0; more && c0 < ncols; c0 += 64) {   // (the first 64 and no more in even patterns)
            const int c = c0 + lane;
            const unsigned long long not_heavy = __ballot(c >= ncols || ranked[list_record(KB, c < ncols ? c : 0)].y <= g.heavy);
            more = not_heavy == 0;
            heavy += more ? 64 : __builtin_ctzll(not_heavy);
        }
        heavy = __builtin_amdgcn_readfirstlane(heavy < ncols / 2 ? heavy : ncols / 2);   // (more only where a list holds more entries than there are blocks)
    }
    const int groups = (ncols + heavy + SP_NC - 1) / SP_NC, more_groups = groups - (ncols + SP_NC - 1) / SP_NC;
    const int tiles = g.tiles[more_groups < SP_MORE ? more_groups : SP_MORE], low_tiles = g.M > tiles * SP_BM ? (g.M - tiles * SP_BM + SP_BM / 2 - 1) / (SP_BM / 2) : 0;

    // The units of this XCD: its share of the tiles x groups, then of the low tiles x groups.  Its workgroups take them in turn, every other round
    // from the other end: who has started with one of the first, which hold the longest columns, does not get the odd one at the end as well.
    const int xcd = blockIdx.x % NUM_XCD, local = blockIdx.x / NUM_XCD, peers = gridDim.x / NUM_XCD;
    auto share = [&](int units, int x) __attribute__((always_inline)) { return (int)((long long)units * x / NUM_XCD); };
    const int full0 = share(tiles * groups, xcd), n_full = share(tiles * groups, xcd + 1) - full0;
    const int low0 = share(low_tiles * groups, xcd), n_low = share(low_tiles * groups, xcd + 1) - low0;
    const int rounds = (n_full + n_low) / peers;
    const int mine = rounds + ((rounds & 1 ? peers - 1 - local : local) < (n_full + n_low) % peers ? 1 : 0);
    if (mine == 0) return;
    // unit j: its group, its first token, and whether its tile is a low one
    auto unit_of = [&](int j, int& group, int& row0, bool& low) __attribute__((always_inline)) {
        const int w = j * peers + (j & 1 ? peers - 1 - local : local);
        low = w >= n_full;
        const int v = low ? low0 + w - n_full : full0 + w, of = low ? low_tiles : tiles;
        const int tb = v / (g.tile_block * groups), rem = v - tb * (g.tile_block * groups);
        int in_block = of - tb * g.tile_block;
        in_block = in_block < g.tile_block ? in_block : g.tile_block;
        group = rem / in_block;
        const int tile = tb * g.tile_block + rem - group * in_block;
        row0 = low ? tiles * SP_BM + tile * (SP_BM / 2) : tile * SP_BM;
    };

    if ((int)threadIdx.x < RS + SP_NC + 1) s_landed[threadIdx.x] = 0;
    __syncthreads();
    bool gave_up = false;
    auto give_up = [&]() __attribute__((always_inline)) {
        gave_up = true;
        if (lane == 0) lds_poke(s_fail, 1);
    };
    auto others_gave_up = [&](int spin) __attribute__((always_inline)) {
        return (spin & 1023) == 1023 && __builtin_amdgcn_readfirstlane(lds_peek(s_fail)) != 0;
    };

    if (wave >= SP_NC) {
        // ---------------- filling the ring: this wave takes the steps p, p + 4, ... ----------------
        const int p = wave - SP_NC;
        const int steps = mine * KB;   // (the host keeps this below 2^30)
        const unsigned stride = (unsigned)g.K * 4u;
        const int row0 = lane >> 3;
        // row 8 i + row0, chunk (lane & 7) / 2 at the chunk ^ (row / 4 % 4): the second term is lane / 32, for odd i with 2 more
        unsigned char* const to = smem + row0 * 64 + (((lane & 7) >> 1) ^ (lane >> 5)) * 16 + (lane & 1) * 8;
        const int to_odd = ((((lane & 7) >> 1) ^ (lane >> 5)) & 2) ? -32 : 32;
        int lj = 0, lkb = p;   // the step being loaded
        while (lkb >= KB) { lkb -= KB; ++lj; }
        unsigned voff[8];
        bool low = false;
        size_t base = 0;   // (offsets from the argument, so that the loads are global and not flat: those would wait for LDS as well)
        const unsigned char* const A = reinterpret_cast<const unsigned char*>(g.a);
        auto set_tile = [&](int j) __attribute__((always_inline)) {
            int group, m0;
            unit_of(j < mine ? j : mine - 1, group, m0, low);
            base = (size_t)m0 * stride;
            int rows = g.M - 1 - m0;   // (rows behind the last one of the tile or the matrix re-read that)
            if (low && rows > SP_BM / 2 - 1) rows = SP_BM / 2 - 1;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int row = 8 * i + row0;
                voff[i] = (unsigned)(row < rows ? row : rows) * stride + (lane & 7) * 16u;
            }
        };
        set_tile(lj);
        float4 buf[2][8];
        bool buf_low[2];
        float buf_scale[2];
        auto load = [&](float4 (&v)[8], bool& v_low, float& v_scale) __attribute__((always_inline)) {
            v_low = low;
            v_scale = with_sign(SP_SCALE, block_sign(lkb));
            const unsigned char* src = A + (base + (size_t)lkb * 128);
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = *reinterpret_cast<const float4*>(src + voff[i]);
            lkb += SP_NP;
            bool moved = false;
            while (lkb >= KB) {
                lkb -= KB;
                ++lj;
                moved = true;
            }
            if (moved) set_tile(lj);
        };
        int s_at = p;   // the slot of the step being filled
        auto fill = [&](int u, const float4 (&v)[8], bool v_low, float v_scale) __attribute__((always_inline)) {
            // split first: a slot that becomes free then only waits for the writes
            uint2 part[3][8];
            auto rows = [&](int i0) __attribute__((always_inline)) {
#pragma unroll
                for (int i = i0; i < i0 + 4; ++i) {
                    split2(v[i].x * v_scale, v[i].y * v_scale, part[0][i].x, part[1][i].x, part[2][i].x);
                    split2(v[i].z * v_scale, v[i].w * v_scale, part[0][i].y, part[1][i].y, part[2][i].y);
                }
            };
            rows(0);
            if (!v_low) rows(4);
            __builtin_amdgcn_sched_barrier(0);
            bool free = false;
            for (int spin = 0; spin < SP_SPIN_LIMIT && !gave_up; ++spin) {
                const int d = lds_peek(s_done + (lane & (SP_NC - 1)));
                free = __all(d > u - RS);
                if (free || others_gave_up(spin)) break;
                __builtin_amdgcn_s_sleep(1);
            }
            if (!free && !gave_up) give_up();
            asm volatile("" ::: "memory");
            unsigned char* slot = to + s_at * SLOT;
            auto write = [&](int i0) __attribute__((always_inline)) {
#pragma unroll
                for (int i = i0; i < i0 + 4; ++i)
#pragma unroll
                    for (int p = 0; p < 3; ++p) *reinterpret_cast<uint2*>(slot + i * 512 + (i & 1 ? to_odd : 0) + p * PLANE) = part[p][i];
            };
            write(0);
            if (!v_low) write(4);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (lane == 0) lds_poke(s_landed + s_at, u + 1);
            s_at = s_at + SP_NP < RS ? s_at + SP_NP : s_at + SP_NP - RS;
        };
        if (p < steps) load(buf[0], buf_low[0], buf_scale[0]);
        for (int u = p; u < steps; u += 2 * SP_NP) {
            load(buf[1], buf_low[1], buf_scale[1]);   // (past the last step: the last tile again, never used)
            fill(u, buf[0], buf_low[0], buf_scale[0]);
            if (u + SP_NP >= steps) break;
            load(buf[0], buf_low[0], buf_scale[0]);
            fill(u + SP_NP, buf[1], buf_low[1], buf_scale[1]);
        }
        if (gave_up) count_protocol_failure();
        return;
    }

    // ---------------- multiplying ----------------
    const int r = lane & 31, h = lane >> 5;
    const int band = wave < 4 ? wave : 11 - wave;   // waves w and w + 4 share a SIMD: a long column and a short one
    const int2* const records = reinterpret_cast<const int2*>(g.plan);
    // block column of the result, its rank, its entries, and first token | (1: the first 32 tokens alone, 2: the second), of this workgroup's units
    struct Head {
        int col, rank, n, row;
    };
    int4* const heads = s_heads + wave * SP_MAX_UNITS;
    if (lane < mine) {
        int group, row0;
        bool low;
        unit_of(lane, group, row0, low);
        const int v = band * groups + ((band & 1) ? groups - 1 - group : group);
        const int rank = v < 2 * heavy ? v >> 1 : v - heavy;
        const int tokens = v >= 2 * heavy ? (low ? 1 : 0) : (v & 1) ? 2 : 1;
        int2 head = make_int2(-1, 0);
        if (rank < ncols && !(low && tokens == 2)) head = records[list_record(KB, rank)];
        heads[lane] = make_int4(head.x, rank < ncols ? rank : 0, head.y, row0 | tokens);
    }
    auto head_of = [&](int j) __attribute__((always_inline)) {
        int4 v = make_int4(-1, 0, 0, 0);
        if (j < mine) v = heads[j];
        return Head{__builtin_amdgcn_readfirstlane(v.x), __builtin_amdgcn_readfirstlane(v.y), __builtin_amdgcn_readfirstlane(v.z), __builtin_amdgcn_readfirstlane(v.w)};
    };

    // The sums of TH times 32 tokens: the column so far, and a block, which joins it when the next one is under way.
    struct Whole {
        f32x16 total[2], part[2];
        int sign;   // of the block in the last part
    };
    struct Half {
        f32x16 total[1], part[1];
        int sign;
    };
    auto join = [&](auto& sums, int t) __attribute__((always_inline)) {
        const float one = with_sign(1.f, sums.sign);
#pragma unroll
        for (int v = 0; v < 16; ++v) sums.total[t][v] = __builtin_fmaf(sums.part[t][v], one, sums.total[t][v]);
    };
    auto clear = [&](auto& sums) __attribute__((always_inline)) {
        sums.sign = 0;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            sums.total[0][v] = sums.part[0][v] = 0.f;
            if constexpr (sizeof(sums) == sizeof(Whole)) sums.total[1][v] = sums.part[1][v] = 0.f;
        }
    };

    auto publish = [&](int u) __attribute__((always_inline)) {
        if (lane == 0) lds_poke(s_done + wave, u);
    };
    auto slot_of = [&](int u) __attribute__((always_inline)) { return (int)((unsigned)u % (unsigned)RS); };
    auto landed = [&](int slot) __attribute__((always_inline)) { return lds_peek(s_landed + slot); };

    auto wait_for = [&](int u) __attribute__((always_inline)) {
        bool here = gave_up;   // after a failed wait nothing is waited for any more: the results are void
        for (int spin = 0; spin < SP_SPIN_LIMIT && !here; ++spin) {
            here = __builtin_amdgcn_readfirstlane(landed(slot_of(u))) > u;
            if (here || others_gave_up(spin)) break;
            __builtin_amdgcn_s_sleep(1);
        }
        if (!here) give_up();
    };
    // results of a unit, a token's 16 values per lane: columns 8 q + 4 h + e of token 32 t + r
    auto epilogue = [&](const Head& unit, auto& sums) __attribute__((always_inline)) {
        constexpr int TH = sizeof(sums) == sizeof(Whole) ? 2 : 1;
        auto& total = sums.total;
        const int col = unit.col, row0 = unit.row & ~3;
        if (col < 0) return;
        join(sums, TH - 1);   // (of the last block)
        const int at = lane_now();   // (the addresses below are made here, not kept in registers while the column is multiplied)
        const int r = at & 31, h = at >> 5;
        const bool failed = gave_up || __builtin_amdgcn_readfirstlane(lds_peek(s_fail)) != 0;
        float b[16];   // (word by word: a bias need not be aligned to more)
#pragma unroll
        for (int v = 0; v < 16; ++v) b[v] = g.bias ? g.bias[col * 32 + 8 * (v >> 2) + 4 * h + (v & 3)] : 0.f;
#pragma unroll
        for (int t = 0; t < TH; ++t) {
            float off = 0.f;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                total[t][v] *= SP_UNSCALE;
                off = __builtin_fmaf(total[t][v], 0.f, off);
            }
            const int row = row0 + (TH == 2 ? t * 32 : (unit.row & 1 ? 0 : 32)) + r;
            if (__any(off != 0.f || off != off)) {
                // again, with fp32 instructions and operands as they are, each block's products summed by themselves as well: infinities, NaN, results
                // beyond the scaled range
                unsigned bad = 0;
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    if (total[t][v] - total[t][v] != 0.f) {
                        bad |= 1u << v;
                        total[t][v] = 0.f;
                    }
                const float* x = g.a + (size_t)(row < g.M ? row : g.M - 1) * g.K;
                const int2* const entries = records + list_record(KB, unit.rank) + LIST_HEAD;
#pragma unroll 1
                for (int i = 0; i < unit.n; ++i) {
                    const int2 e = entries[i];
                    const float* w = g.data + (size_t)e.y * 1024 + (TRANS ? r * 32 + 16 * h : 16 * h * 32 + r);
                    f32x16 s;
#pragma unroll
                    for (int v = 0; v < 16; ++v) s[v] = 0.f;
#pragma unroll 1
                    for (int k0 = 0; k0 < 16; k0 += 8) {
                        float wk[8], xk[8];   // k = 16 h + k0 + 0 .. 7, asked for together
#pragma unroll
                        for (int k = 0; k < 8; ++k) {
                            wk[k] = w[(k0 + k) * (TRANS ? 1 : 32)];
                            xk[k] = x[e.x * 32 + 16 * h + k0 + k];
                        }
#pragma unroll
                        for (int k = 0; k < 8; ++k) s = __builtin_amdgcn_mfma_f32_32x32x2f32(wk[k], xk[k], s, 0, 0, 0);
                    }
#pragma unroll
                    for (int v = 0; v < 16; ++v) total[t][v] = bad >> v & 1 ? total[t][v] + s[v] : total[t][v];
                }
            }
            if (row < g.M) {
                float* o = g.out + (size_t)row * g.N + col * 32 + 4 * h;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float4 v = make_float4(total[t][4 * q] + b[4 * q], total[t][4 * q + 1] + b[4 * q + 1], total[t][4 * q + 2] + b[4 * q + 2], total[t][4 * q + 3] + b[4 * q + 3]);
                    if (failed) v.x = v.y = v.z = v.w = __builtin_nanf("");
                    *reinterpret_cast<float4*>(o + 8 * q) = v;
                }
            }
        }
    };

    // the entries i0 .. i0 + 63 of a unit's column, one per lane.  Of a column without blocks, or behind the last unit, the first k-block and block 0: both
    // exist, no step of the ring that is still needed is given up for them, and nothing is read of the plan, whose entries no list may have written.
    auto window = [&](const Head& unit, int i0) __attribute__((always_inline)) {
        int2 e = make_int2(0, 0);
        if (unit.n > 0) {
            const int l = i0 + lane_now();
            e = records[list_record(KB, unit.rank) + LIST_HEAD + (l < unit.n ? l : unit.n - 1)];
        }
        return e;
    };
    auto arrived = [](int2& w) __attribute__((always_inline)) { asm volatile("" : "+v"(w.x), "+v"(w.y)); };
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    u32x4 first[6];   // [k half][part] of the block that a unit starts with
    const unsigned lane16 = lane * 16u;
    auto load_block = [&](u32x4 (&w)[6], int b) __attribute__((always_inline)) {
        const unsigned char* src = g.parts + (size_t)(unsigned)b * SP_BLOCK_BYTES;
#pragma unroll
        for (int i = 0; i < 6; ++i) w[i] = *reinterpret_cast<const u32x4*>(src + i * 1024 + lane16);
    };
    // chunk c (8 values of k) of token row r at c ^ (r / 4 % 4): 16 rows' reads of one chunk meet no bank twice
    const unsigned x_at = r * 64 + ((h ^ ((r >> 2) & 3)) * 16);   // (the other half of k: ^ 32)

    // entries of this unit and the next, and those of the one after, on their way
    Head unit = head_of(0);
    int2 ev = window(unit, 0), ev1 = window(head_of(1), 0), ev2 = make_int2(0, 0);
    arrived(ev);
    arrived(ev1);
    load_block(first, __builtin_amdgcn_readlane(ev.y, 0));
    int raw = 0, slot = 0;
    for (int j = 0; j < mine; ++j) {
        const int n = unit.n, u0 = j * KB;
        if (n > 0) {
            int kb = __builtin_amdgcn_readlane(ev.x, 0);
            publish(u0 + kb);
            slot = slot_of(u0 + kb);
            int i = 0;
            if (unit.row & 3) {
                // A wave with 32 tokens of the tile: an item is shorter than a block's way from the L2, and waiting for its operands would be a third of it.  The
                // registers of the other 32 tokens are free: blocks are asked for two items ahead, and an operand is read for the next item once it is used.  On a
                // path of its own (the choice cost the whole tiles 1.3 %): 28 products with Zipf rows 1.045 times as fast forward, 1.014 input gradient, up to 1.12
                // (1824 -> 1472 density 0.667, 2720 tokens 86 -> 77 us).  The same for whole tiles, and filling waves that wait for no LDS access they have just
                // made, give nothing (0.98 to 1.0): these kernels are bound by power, and the clock gives back what their cycles save.
                Half sums;
                clear(sums);
                u32x4 x[2][3];   // [half of k][part]
                const unsigned x_half = x_at + (unit.row & 1 ? 0 : 2048);
                auto read = [&](int q, int p) __attribute__((always_inline)) {
                    x[q][p] = *reinterpret_cast<const u32x4*>(smem + ((q ? x_half ^ 32 : x_half) + slot * SLOT) + p * PLANE);
                };
                auto here = [&]() __attribute__((always_inline)) {
                    if (__builtin_expect(__builtin_amdgcn_readfirstlane(raw) <= u0 + kb, 0)) wait_for(u0 + kb);
                    asm volatile("" ::: "memory");
                };
                int kb_next = 0;
                auto entry = [&](int i, int& at, int& b) __attribute__((always_inline)) {   // (behind the last one the first of the next unit)
                    const bool inside = i < n;
                    if ((i & 63) == 0 && inside) {
                        ev = window(unit, i);
                        arrived(ev);
                    }
                    const int kb_in = __builtin_amdgcn_readlane(ev.x, i & 63), kb_out = KB + __builtin_amdgcn_readlane(ev1.x, 0);
                    const int b_in = __builtin_amdgcn_readlane(ev.y, i & 63), b_out = __builtin_amdgcn_readlane(ev1.y, 0);
                    at = inside ? kb_in : kb_out;
                    b = inside ? b_in : b_out;
                };
                auto item = [&](int i, const u32x4 (&w)[6], u32x4 (&w_ahead)[6]) __attribute__((always_inline)) {
                    const bool more = i + 1 < n;
                    int kb_ahead, b_ahead;
                    entry(i + 2, kb_ahead, b_ahead);
                    const int this_sign = block_sign(kb);
                    load_block(w_ahead, b_ahead);
                    kb = kb_next;
                    kb_next = kb_ahead;
                    slot = slot_of(u0 + kb);
                    __builtin_amdgcn_sched_barrier(0);
                    join(sums, 0);   // the block before
                    sums.sign = this_sign;
                    asm volatile("" : "+v"(sums.total[0]));
#pragma unroll
                    for (int v = 0; v < 16; ++v) sums.part[0][v] = 0.f;
                    auto mma = [&](int q, int pw, int px) __attribute__((always_inline)) {
                        sums.part[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w[3 * q + pw]), __builtin_bit_cast(bf16x8, x[q][px]),
                                                                               sums.part[0], 0, 0, 0);
                    };
                    mma(0, 0, 2);
                    mma(0, 1, 1);
                    mma(0, 0, 1);
                    __builtin_amdgcn_sched_barrier(0);
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // every read of the slot
                    publish(u0 + kb);   // (behind the last item this may be less than the next unit needs, never more)
                    raw = landed(slot);
                    __builtin_amdgcn_sched_barrier(0);
                    mma(0, 2, 0);
                    mma(0, 1, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (more) {
                        here();
                        read(0, 2);
                        read(0, 1);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    mma(1, 0, 2);
                    mma(1, 1, 1);
                    mma(1, 0, 1);
                    mma(1, 2, 0);
                    mma(1, 1, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (more) {
                        read(1, 2);
                        read(1, 1);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    mma(0, 0, 0);
                    mma(1, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    if (more) {
                        read(0, 0);
                        read(1, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                };
                u32x4 w0[6], w1[6], w2[6];
                here();
#pragma unroll
                for (int k = 0; k < 6; ++k) read(k / 3, 2 - k % 3);
#pragma unroll
                for (int k = 0; k < 6; ++k) w0[k] = first[k];
                int b_next;
                entry(1, kb_next, b_next);
                load_block(w1, b_next);
                while (true) {
                    item(i, w0, w2);
                    if (++i == n) {
#pragma unroll
                        for (int k = 0; k < 6; ++k) first[k] = w1[k];
                        break;
                    }
                    item(i, w1, w0);
                    if (++i == n) {
#pragma unroll
                        for (int k = 0; k < 6; ++k) first[k] = w2[k];
                        break;
                    }
                    item(i, w2, w1);
                    if (++i == n) {
#pragma unroll
                        for (int k = 0; k < 6; ++k) first[k] = w0[k];
                        break;
                    }
                }
                ev2 = window(head_of(j + 2), 0);
                epilogue(unit, sums);
            } else {
                Whole sums;
                clear(sums);
                // one item: w = its block, w_next takes the next one's (behind the last one the first of the next unit)
                auto item = [&](int i, u32x4 (&w)[6], u32x4 (&w_next)[6]) __attribute__((always_inline)) {
                    const int u = u0 + kb;
                    const int this_sign = block_sign(kb);
                    const bool last = i + 1 == n;
                    if (((i + 1) & 63) == 0 && !last) {
                        ev = window(unit, i + 1);
                        arrived(ev);
                    }
                    const int kb_in = __builtin_amdgcn_readlane(ev.x, (i + 1) & 63), kb_out = KB + __builtin_amdgcn_readlane(ev1.x, 0);
                    kb = last ? kb_out : kb_in;
                    const int b_in = __builtin_amdgcn_readlane(ev.y, (i + 1) & 63), b_out = __builtin_amdgcn_readlane(ev1.y, 0);
                    load_block(w_next, last ? b_out : b_in);
                    if (__builtin_expect(__builtin_amdgcn_readfirstlane(raw) <= u, 0)) wait_for(u);
                    asm volatile("" ::: "memory");
                    const unsigned char* p0 = smem + (x_at + slot * SLOT);
                    const unsigned char* p1 = smem + ((x_at ^ 32) + slot * SLOT);
                    u32x4 x[2][3];   // [half of k][part] of 32 tokens
                    auto read = [&](int t, int q, int p) __attribute__((always_inline)) {
                        x[q][p] = *reinterpret_cast<const u32x4*>((q ? p1 : p0) + p * PLANE + t * 2048);
                    };
#pragma unroll
                    for (int k = 0; k < 6; ++k) read(0, k / 3, 2 - k % 3);
                    slot = slot_of(u0 + kb);
                    auto reads_back = [&]() __attribute__((always_inline)) {   // every read of the slot
                        raw = landed(slot);
                        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                        publish(u0 + kb);   // (behind the last item this may be less than the next unit needs, never more)
                    };
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        f32x16& c = sums.part[t];
                        auto mma = [&](int q, int pw, int px) __attribute__((always_inline)) {
                            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w[3 * q + pw]), __builtin_bit_cast(bf16x8, x[q][px]), c, 0, 0, 0);
                        };
                        auto small = [&](int q) __attribute__((always_inline)) {   // (first those whose operands are read first)
                            mma(q, 0, 2);
                            mma(q, 1, 1);
                            mma(q, 0, 1);
                            mma(q, 2, 0);
                            mma(q, 1, 0);
                        };
#pragma unroll
                        for (int v = 0; v < 16; ++v) c[v] = 0.f;
                        small(0);
                        __builtin_amdgcn_sched_barrier(0);
                        if (t == 0) {
                            read(1, 0, 2);
                            read(1, 0, 1);
                        }
                        join(sums, t ^ 1);   // t = 0: of the block before
                        if (t == 0) sums.sign = this_sign;
                        asm volatile("" : "+v"(sums.total[t ^ 1]));   // (here, where matrix instructions are under way, and not at the end)
                        __builtin_amdgcn_sched_barrier(0);
                        small(1);
                        mma(0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                        if (t == 0) {
                            read(1, 0, 0);
                            read(1, 1, 2);
                            read(1, 1, 1);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                        mma(1, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                        if (t == 0) {
                            read(1, 1, 0);
                            reads_back();
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                };
                u32x4 w1[6];
                bool odd;
                while (true) {
                    item(i, first, w1);
                    odd = true;
                    if (++i == n) break;
                    item(i, w1, first);
                    odd = false;
                    if (++i == n) break;
                }
                ev2 = window(head_of(j + 2), 0);
                epilogue(unit, sums);
                if (odd) {
#pragma unroll
                    for (int k = 0; k < 6; ++k) first[k] = w1[k];
                }
            }
        } else {
            ev2 = window(head_of(j + 2), 0);
            if (unit.row & 3) {
                Half sums;
                clear(sums);
                epilogue(unit, sums);
            } else {
                Whole sums;
                clear(sums);
                epilogue(unit, sums);
            }
            if (j + 1 < mine) load_block(first, __builtin_amdgcn_readlane(ev1.y, 0));
        }
        arrived(ev2);
        unit = head_of(j + 1);
        ev = ev1;
        ev1 = ev2;
    }
    publish(0x7fffffff);
    if (gave_up) count_protocol_failure();
}

}  // namespace pbs
