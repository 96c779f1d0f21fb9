// dense x block-sparse -> dense for bf16 with a short contraction (K <= 1024): the workgroup's token tile stays in LDS.
//
// A workgroup of 16 waves copies its 64 tokens, all K features of them, into LDS once, in whole rows; after one barrier each
// wave multiplies block columns of its own, one after the other, and nothing is shared but the tile, which nobody writes any
// more: no progress words, no further barrier, and a column costs what it holds.  A wave's block (2 KB) passes through LDS of
// its own like in pbs_stream.h: DMA, fragments into registers, and the place takes the next block's DMA, of the next
// column too.
//
// Why: the stream kernel fetches the token tile again for every block (10 KB per block and 128 tokens, in rows of 64 bytes, is
// what bounds it), the wide kernel (pbs_dds16.h) moves panels through a ring and pays for every step of it.  Here a
// block costs 2 KB of copies and 64 tokens' fragments from LDS, and four waves per SIMD keep the matrix cores near their rate
// while they multiply: a block takes 128 cycles of a SIMD, which is what its matrix instructions take.  What is left around that:
// launch, list and tile (4 to 6 us), and the stores, which bound wide results (768 -> 3072 at 16384 tokens writes 100 MB).
// One block at a time per wave: a second place in the ring is 3 to 7 % slower (its LDS, and two loads in flight per wave
// are not needed with four waves per SIMD); tiles of 32 tokens are 20 to 60 % slower from 2000 tokens (twice the copies).
//
// Measured, us, against what ran before: 768 -> 3072 density 0.5, 2317 tokens 22.9 -> 13.7 (stream), 4096 tokens 29.6 -> 19.5,
// 16384 tokens 123 -> 53.5 (wide); 768 -> 3072 density 0.1, 16384 tokens 40 -> 28; 768 -> 768 density 0.5, 16384 tokens
// 25.8 -> 20.6; 992 -> 2016 density 0.5, 16384 tokens 92 -> 46.  Below some thousand tokens, or with few columns, the stream
// kernel is the faster one (768 -> 768, 2317 tokens 8.3 against 9.7).
#pragma once
#include "pbs_common.h"
#include "pbs_stream.h"

namespace pbs {

constexpr int PANEL_NW = 16;          // waves of a workgroup
constexpr int PANEL_TT = 4;           // token tile in units of 16
constexpr int PANEL_MAX_K = 1024;     // 160 KB of LDS: the tile and a block per wave; a column's list fits half a wave

struct PanelArgs {
    const void* a;      // [M, K] row-major
    const void* data;   // [nnz*32, 32]
    const int* plan;    // the list plan
    const void* bias;   // nullptr or [N]
    void* out;          // [M, N] row-major
    int M, N, K;
    int splits;         // workgroups that share a token tile: every splits-th column of the ranking each
};

// a row of the tile in LDS, in 16-byte chunks: whole groups of 16 (256 bytes), so that the swizzle stays inside a group
static inline __host__ __device__ int panel_chunks(int K) { return (K / 8 + 15) / 16 * 16; }
static inline size_t panel_lds(int K) { return (size_t)16 * PANEL_TT * panel_chunks(K) * 16 + (size_t)PANEL_NW * 2048; }

// TRANS as in stream_kernel.
template <int TRANS>
__global__ __launch_bounds__(PANEL_NW * 64, 4) void panel_kernel(PanelArgs g) {
    using E = Elem<bf16_t>;
    constexpr int TT = PANEL_TT, BM = 16 * TT, NW = PANEL_NW;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    const int ncols = g.N >> 5;
    const int tiles = (g.M + BM - 1) / BM;
    const int id = xcd_tile_id(blockIdx.x, tiles * g.splits);
    if (id < 0) return;
    const int tile = id / g.splits, split = id - tile * g.splits;
    const int m0 = tile * BM;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4;

    const int ckp = panel_chunks(g.K), pitch = ckp * 16;
    const unsigned char* A = static_cast<const unsigned char*>(g.a) + (size_t)m0 * g.K * 2;
    const unsigned char* D = static_cast<const unsigned char*>(g.data);
    const unsigned lds0 = (unsigned)(uintptr_t)smem;
    unsigned char* const place = smem + BM * pitch + wave * 2048;   // this wave's block
    const unsigned lds_place = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)place);

    // ---- the token tile: chunk p of row t holds chunk p ^ (t % 16) of the row, so that 16 rows' reads of one chunk meet no bank twice ----
    {
        const int rows = g.M - m0 < BM ? g.M - m0 : BM, last = g.K / 8 - 1;
        for (int i = wave; i < BM * ckp / 64; i += NW) {
            const int at = i * 64 + lane, t = at / ckp;
            int c = (at - t * ckp) ^ (t & 15);
            c = c < last ? c : last;
            dma16(__builtin_amdgcn_readfirstlane(lds0 + i * 1024), A, (unsigned)((t < rows ? t : rows - 1) * (g.K * 2) + c * 16));
        }
    }

    // ---- this wave's columns: of the workgroup's (ranked by length) one in each run of NW, the runs taken forth and back ----
    const int nc = (ncols - split + g.splits - 1) / g.splits;
    auto turn = [&](int i) { return i * NW + (i & 1 ? NW - 1 - wave : wave); };
    int mine = nc / NW;
    if (turn(mine) < nc) ++mine;
    const int pairs = (mine + 1) / 2;
    // two columns at a time, one per half of the wave: lane l has the half's column, its length, entry l % 32 and bias l % 32
    struct Pair {
        int n, col;
        int2 e;
        float b;
    };
    const int KB = g.K >> 5;
    auto load_pair = [&](int p) {
        Pair o{0, 0, make_int2(0, 0), 0.f};
        const int i = 2 * p + (lane >> 5), l = lane & 31;
        if (i < mine) {
            // (the entry with the head: places behind the last one hold anything, and are not multiplied)
            const int2* record = reinterpret_cast<const int2*>(g.plan) + list_record(KB, split + g.splits * turn(i));
            const int2 head = record[0];
            const int2 e = record[LIST_HEAD + (l < KB ? l : KB - 1)];
            o.n = head.y < 32 ? head.y : 32;
            o.col = head.x;
            if (l < o.n) o.e = e;
            if (g.bias) o.b = E::to_f32(static_cast<const bf16_t*>(g.bias)[head.x * 32 + l]);
        }
        return o;
    };
    Pair cur = load_pair(0), nxt = load_pair(1);
    float bias_of[2] = {cur.b, 0.f};   // by pair % 2

    auto w_row_swz = [](int row) { return (row >> 3) & 3; };
    unsigned w_voff[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = i * 16 + lane / 4;
        w_voff[i] = TRANS ? row * 64 + ((lane & 3) ^ w_row_swz(row)) * 16 : i * 1024 + lane * 16;
    }

    // ---- the blocks in the order they are multiplied, asked for one ahead ----
    constexpr int LAST = 1, EMPTY = 2, HALF = 4, ODD = 8, VALID = 16;
    int kb = 0, col = 0, what = 0;   // the block asked for: k-block, block column, flags
    int pair = 0, half = 0, idx = 0;
    auto ask = [&]() __attribute__((always_inline)) {
        what = 0;
        if (pair >= pairs) return;
        const int src = half * 32;
        const int n = __builtin_amdgcn_readlane(cur.n, src);
        col = __builtin_amdgcn_readlane(cur.col, src);
        kb = __builtin_amdgcn_readlane(cur.e.x, src + idx);
        // (a column without blocks asks for some block and does not multiply it)
        const unsigned char* pw = uniform_ptr(D + (size_t)__builtin_amdgcn_readlane(cur.e.y, src + idx) * 2048);
        dma16(lds_place, pw, w_voff[0]);
        dma16(lds_place + 1024, pw, w_voff[1]);
        const bool end = idx + 1 >= n;
        what = VALID | (end ? LAST : 0) | (n == 0 ? EMPTY : 0) | (half ? HALF : 0) | (pair & 1 ? ODD : 0);
        ++idx;
        if (end) {
            idx = 0;
            ++half;
            if (half == 2 || 2 * pair + half >= mine) {
                half = 0;
                ++pair;
                cur = nxt;
                nxt = load_pair(pair + 1);
                if (pair & 1) bias_of[1] = cur.b;
                else bias_of[0] = cur.b;
            }
        }
    };
    ask();

    drain_barrier();   // the tile is there

    f32x4 acc[TT][2];
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[t][0] = acc[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    const unsigned char* a_row = smem + r * pitch;
    while (what & VALID) {
        wait_dma(0);
        uint4 fa[TT], fw[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if constexpr (TRANS) {
                const int row = 8 * (r >> 2) + 4 * j + (r & 3);
                fw[j] = *reinterpret_cast<const uint4*>(place + row * 64 + (q ^ w_row_swz(row)) * 16);
            } else {
                const unsigned char* p = place + (8 * q + (r >> 2)) * 64 + (r & 3) * 16 + 8 * j;
                const uint2 lo = tr16_b64(p), hi = tr16_b64(p + 256);
                fw[j] = make_uint4(lo.x, lo.y, hi.x, hi.y);
            }
        }
        const unsigned char* as = a_row + (((kb * 4 + q) ^ r) * 16);
#pragma unroll
        for (int t = 0; t < TT; ++t) fa[t] = *reinterpret_cast<const uint4*>(as + 16 * t * pitch);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const int now = what;
        const size_t out_col = (size_t)col * 32 + 8 * q;
        const float b = now & ODD ? bias_of[1] : bias_of[0];   // (before the next pair but one may replace it)
        ask();
        if (!(now & EMPTY)) {
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, fw[j]), __builtin_bit_cast(bf16x8, fa[t]), acc[t][j], 0, 0, 0);
        }
        if (now & LAST) {
            // a lane's eight results of a token: columns 8 q .. 8 q + 7, four of each parity
            float bv[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) bv[i] = __shfl(b, (now & HALF ? 32 : 0) + 8 * q + i, 64);
            uint16_t* out = static_cast<uint16_t*>(g.out) + out_col;
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                const int row = m0 + 16 * t + r;
                uint32_t w[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float v0 = acc[t][i >> 1][2 * (i & 1)] + bv[2 * i], v1 = acc[t][i >> 1][2 * (i & 1) + 1] + bv[2 * i + 1];
                    w[i] = (uint32_t)E::from_f32(v0).bits | ((uint32_t)E::from_f32(v1).bits << 16);
                }
                if (row < g.M) *reinterpret_cast<uint4*>(out + (size_t)row * g.N) = make_uint4(w[0], w[1], w[2], w[3]);
                acc[t][0] = acc[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
    }
}

// The same for contractions that do not fit: the tile passes through LDS in chunks of 512 features, two buffers, the next chunk on its way
// while this one is multiplied, one barrier per chunk.  A column belongs to S waves (every S-th of its blocks each), whose sums meet
// in LDS at the end; one column per wave, so the accumulators stay where they are from chunk to chunk.  S = 4, 2, 1 make 4, 8, 16 columns per
// workgroup: few tokens need many workgroups, many tokens fewer that share a tile.  The lists are by k-block (list_plan).
//
// What bounds it: a chunk's copy, 64 KB at the texture path's rate (1.5 k cycles) and its latency behind the barrier (0.8 us per chunk in all).
// Measured, us, against the stream kernel: 3072 -> 768 density 0.5, 2317 tokens 21.8 -> 16.5, 4096 tokens 27.8 -> 22.7; 4096 -> 4096
// density 0.25, 1024 tokens 30.3 -> 24.1; 4096 -> 1024 density 0.75, 4096 tokens 69.8 -> 36.7; 1536 -> 2976 density 0.4, 2317 tokens
// 31.8 -> 20.1.  With fewer tokens and columns it is the slower one (3072 -> 768, 509 tokens 7.6 against 12.2).
constexpr int PANEL_KC = 512;         // features of a chunk: 64 rows of 1 KB
constexpr int PANEL_CHUNK_LDS = 2 * 16 * PANEL_TT * 1024 + PANEL_NW * 2048;
template <int TRANS, int S>
__global__ __launch_bounds__(PANEL_NW * 64, 4) void panel_chunk_kernel(PanelArgs g) {
    using E = Elem<bf16_t>;
    constexpr int TT = PANEL_TT, BM = 16 * TT, NW = PANEL_NW, BUF = BM * 1024, KBC = PANEL_KC / 32;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    const int ncols = g.N >> 5;
    const int tiles = (g.M + BM - 1) / BM;
    const int id = xcd_tile_id(blockIdx.x, tiles * g.splits);
    if (id < 0) return;
    const int tile = id / g.splits, split = id - tile * g.splits;
    const int m0 = tile * BM;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4;
    const int s = wave % S;
    const int rank = split + g.splits * (wave / S);

    const unsigned char* A = static_cast<const unsigned char*>(g.a) + (size_t)m0 * g.K * 2;
    const unsigned char* D = static_cast<const unsigned char*>(g.data);
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)smem);
    unsigned char* const place = smem + 2 * BUF + wave * 2048;   // this wave's block
    const unsigned lds_place = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)place);

    const int rows = g.M - m0 < BM ? g.M - m0 : BM, last_chunk = g.K / 8 - 1;
    const int nchunks = (g.K + PANEL_KC - 1) / PANEL_KC;
    // place p of row t of a chunk holds 16-byte piece p ^ (t % 16)
    auto stage = [&](int ci) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < BM / NW; ++k) {
            const int t = wave + k * NW;
            int c = ci * (PANEL_KC / 8) + (lane ^ (t & 15));
            c = c < last_chunk ? c : last_chunk;
            dma16(lds0 + (ci & 1) * BUF + t * 1024, A, (unsigned)((t < rows ? t : rows - 1) * (g.K * 2) + c * 16));
        }
    };
    stage(0);

    const int KB = g.K >> 5;
    const int2* const record = reinterpret_cast<const int2*>(g.plan) + list_record(KB, rank < ncols ? rank : 0);
    const int2* const ent = record + LIST_HEAD + s;
    const int room = (KB - 1 - s) / S;   // (the record's last place for an entry of this wave's: there are more than PANEL_MAX_K / 32 k-blocks)
    int2 ev = ent[(size_t)(lane < room ? lane : room) * S];   // (with the head: places behind the last entry hold anything, and are not asked for)
    const int2 head = record[0];
    const int n = rank < ncols ? __builtin_amdgcn_readfirstlane(head.y) : 0;
    const int col = rank < ncols ? __builtin_amdgcn_readfirstlane(head.x) * 32 : 0;
    const int mine = n > s ? (n - s + S - 1) / S : 0;
    auto load64 = [&](int i) { return ent[(size_t)(i + lane < mine ? i + lane : mine - 1) * S]; };
    float bv[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) bv[i] = g.bias ? E::to_f32(static_cast<const bf16_t*>(g.bias)[col + 8 * q + i]) : 0.f;

    auto w_row_swz = [](int row) { return (row >> 3) & 3; };
    unsigned w_voff[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int row = i * 16 + lane / 4;
        w_voff[i] = TRANS ? row * 64 + ((lane & 3) ^ w_row_swz(row)) * 16 : i * 1024 + lane * 16;
    }
    int kb = 1 << 30;   // k-block of the block asked for; none: past every chunk
    auto ask = [&](int i) __attribute__((always_inline)) {
        kb = 1 << 30;
        if (i >= mine) return;
        if (i > 0 && (i & 63) == 0) ev = load64(i);
        kb = __builtin_amdgcn_readlane(ev.x, i & 63);
        const unsigned char* pw = uniform_ptr(D + (size_t)__builtin_amdgcn_readlane(ev.y, i & 63) * 2048);
        dma16(lds_place, pw, w_voff[0]);
        dma16(lds_place + 1024, pw, w_voff[1]);
    };
    int i = 0;
    ask(0);

    f32x4 acc[TT][2];
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[t][0] = acc[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int ci = 0; ci < nchunks; ++ci) {
        drain_barrier();   // chunk ci and this wave's block are there, and every wave has left the other buffer
        if (ci + 1 < nchunks) stage(ci + 1);
        const unsigned char* a_row = smem + (ci & 1) * BUF + r * 1024;
        for (bool first = true; kb < (ci + 1) * KBC; first = false) {
            if (!first) wait_dma(0);
            uint4 fa[TT], fw[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                if constexpr (TRANS) {
                    const int row = 8 * (r >> 2) + 4 * j + (r & 3);
                    fw[j] = *reinterpret_cast<const uint4*>(place + row * 64 + (q ^ w_row_swz(row)) * 16);
                } else {
                    const unsigned char* p = place + (8 * q + (r >> 2)) * 64 + (r & 3) * 16 + 8 * j;
                    const uint2 lo = tr16_b64(p), hi = tr16_b64(p + 256);
                    fw[j] = make_uint4(lo.x, lo.y, hi.x, hi.y);
                }
            }
            const int at = kb > ci * KBC ? kb - ci * KBC : 0;   // (inside the chunk whatever the list holds)
            const unsigned char* as = a_row + (((at * 4 + q) ^ r) * 16);
#pragma unroll
            for (int t = 0; t < TT; ++t) fa[t] = *reinterpret_cast<const uint4*>(as + 16 * t * 1024);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            ask(++i);
#pragma unroll
            for (int t = 0; t < TT; ++t)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, fw[j]), __builtin_bit_cast(bf16x8, fa[t]), acc[t][j], 0, 0, 0);
        }
    }

    auto store = [&](int t, const f32x4& v0, const f32x4& v1) __attribute__((always_inline)) {
        const int row = m0 + 16 * t + r;
        if (row >= g.M || rank >= ncols) return;
        uint32_t w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const f32x4& v = e < 2 ? v0 : v1;
            w[e] = (uint32_t)E::from_f32(v[2 * (e & 1)] + bv[2 * e]).bits | ((uint32_t)E::from_f32(v[2 * (e & 1) + 1] + bv[2 * e + 1]).bits << 16);
        }
        *reinterpret_cast<uint4*>(static_cast<uint16_t*>(g.out) + (size_t)row * g.N + col + 8 * q) = make_uint4(w[0], w[1], w[2], w[3]);
    };
    if constexpr (S == 1) {
#pragma unroll
        for (int t = 0; t < TT; ++t) store(t, acc[t][0], acc[t][1]);
    } else {
        f32x4* red = reinterpret_cast<f32x4*>(smem);   // [wave][t][j][lane]: the two buffers
        static_assert(NW * TT * 2 * 1024 <= 2 * BUF, "the sums fit the buffers");
        drain_barrier();
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int j = 0; j < 2; ++j) red[((wave * TT + t) * 2 + j) * 64 + lane] = acc[t][j];
        lds_barrier();
        for (int t = s; t < TT; t += S) {
            f32x4 v[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                v[j] = red[(((wave - s) * TT + t) * 2 + j) * 64 + lane];
#pragma unroll
                for (int w = 1; w < S; ++w) v[j] += red[(((wave - s + w) * TT + t) * 2 + j) * 64 + lane];
            }
            store(t, v[0], v[1]);
        }
    }
}

}  // namespace pbs
