// dense x block-sparse -> dense in fp32 for many token tiles: one wave per block column and run of tiles.
//
// stream_kernel (pbs_stream.h) starts a workgroup per token tile and column: list, first operands, a few blocks, the sum of its waves in LDS, the stores. The workgroups of a CU
// begin together and do all that in step, so with few blocks to a column the matrix cores have work for half of the time (2240 -> 1920 density 0.085, 12337 tokens: busy
// 0.51 of it at 2.3 GHz, a sixth of it lost at the start and the end).  Here a wave takes its column alone, for one to three token tiles of 32, one after the other: the list is
// read once, the next tile's first operands are on their way while the last block of this one is multiplied, and nothing is shared between waves, so there are no barriers.
// The column's blocks go to SUMS sums in turn, which are added like those of stream_kernel's waves: a token's result has the same bits as there.
//
// What bounds it: the texture path (8 KB per block, 0.87 of the cycles of its matrix instructions) and memory.  Tiles of 64 tokens copy 12 KB for twice the
// products, but 12 KB and 162 registers a wave leave three waves to a SIMD: 2 to 20 % slower; of 48 tokens between the two, of 16 5 to 15 % slower, of 128 spilled.
// Measured, us, stream_kernel -> here: 608 -> 1248 density 0.1, 12843 tokens 37.5 -> 29.2; 256 -> 1792 density 0.16, 13092 tokens 38.6 -> 31.0; 1184 -> 2880 density
// 0.07, 4682 tokens 36.4 -> 30.7; 768 -> 3040 density 0.16, 15769 tokens 148 -> 128; 448 -> 640 density 0.46, 14976 tokens 45.3 -> 41.6; 2240 -> 1920 above 113 -> 104.
#pragma once
#include <type_traits>

#include "pbs_common.h"
#include "pbs_stream.h"

namespace pbs {

constexpr int WALK_TT = 2;   // token tile in units of 16
struct WalkArgs {
    StreamArgs s;
    int run;   // token tiles of a wave
};

// TRANS as in stream_kernel; SUMS: its number of waves.
template <int TRANS, int SUMS>
__global__ __launch_bounds__(64, SUMS == 2 ? 4 : 3) void walk_kernel(WalkArgs w) {
    using C = StreamCfg<float, TRANS, WALK_TT, 1>;
    constexpr int TT = WALK_TT, BM = C::BM, NV = 2 * TT;
    const StreamArgs& g = w.s;
    __shared__ __attribute__((aligned(1024))) unsigned char smem[C::SLOT];

    const int ncols = g.N >> 5, KB = g.K >> 5;
    const int xcd = blockIdx.x % NUM_XCD, local = blockIdx.x / NUM_XCD;
    const int xt = xcd % g.xcd_t, xc = xcd / g.xcd_t, cstep = NUM_XCD / g.xcd_t;
    // this XCD: token tiles t_lo .. t_hi - 1 in runs, ranked columns xc, xc + cstep, ...
    const int t_lo = (int)((long long)g.m_tiles * xt / g.xcd_t), t_hi = (int)((long long)g.m_tiles * (xt + 1) / g.xcd_t);
    const int runs = (t_hi - t_lo + w.run - 1) / w.run;
    const int nc = (ncols - xc + cstep - 1) / cstep;
    if (local >= runs * nc) return;
    const int gsz = g.group * nc;   // (group: runs that share one pass over the columns)
    const int grp = local / gsz, rem = local - grp * gsz;
    int tg = runs - grp * g.group;
    tg = tg < g.group ? tg : g.group;
    const int ci = rem / tg;
    const int cr = xc + ci * cstep;
    const int first = t_lo + (grp * g.group + rem - ci * tg) * w.run;
    const int end_tile = first + w.run < t_hi ? first + w.run : t_hi;

    const int lane = threadIdx.x & 63;
    const int r = lane & 15, q = lane >> 4;
    const int2* const record = reinterpret_cast<const int2*>(g.plan) + list_record(KB, cr);
    const int2* const ent = record + LIST_HEAD;
    int2 ev = ent[lane < KB ? lane : KB - 1];
    const int2 head = record[0];
    const int n = __builtin_amdgcn_readfirstlane(head.y);
    const int col = __builtin_amdgcn_readfirstlane(head.x) * 32;
    const float bias = g.bias ? static_cast<const float*>(g.bias)[col + (lane & 31)] : 0.f;   // of column lane % 32

    const unsigned char* const A = static_cast<const unsigned char*>(g.a);
    const unsigned char* const D = static_cast<const unsigned char*>(g.data);
    const unsigned lds_slot = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)smem);
    const unsigned row_bytes = (unsigned)g.K * 4u;

    unsigned a_voff[C::A_DMA];
    auto rows_of = [&](int tile) __attribute__((always_inline)) {   // (tokens behind the last one re-read that)
        const int left = g.M - 1 - tile * BM;
#pragma unroll
        for (int i = 0; i < C::A_DMA; ++i) {
            const int row = i * C::RPI + lane / 8, chunk = (lane & 7) ^ chunk_swz<8>(row);
            a_voff[i] = (unsigned)(row < left ? row : left) * row_bytes + chunk * 16;
        }
    };
    rows_of(first);
    auto w_row_swz = [](int row) { return (row >> 1) & 7; };
    unsigned w_voff[C::W_DMA];
#pragma unroll
    for (int i = 0; i < C::W_DMA; ++i) {
        const int row = i * 8 + lane / 8;
        if constexpr (TRANS) w_voff[i] = row * 128 + ((lane & 7) ^ w_row_swz(row)) * 16;
        else w_voff[i] = ((row & 16) + 4 * (row & 3) + ((row >> 2) & 3)) * 128 + (lane & 7) * 16;
    }

    f32x4 acc[SUMS][TT][2];
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < SUMS; ++s)
#pragma unroll
            for (int t = 0; t < TT; ++t) acc[s][t][0] = acc[s][t][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    clear();

    constexpr int NISSUE = C::A_DMA + C::W_DMA;
    const unsigned char *pa = nullptr, *pw = nullptr;   // the operands being asked for
    auto source = [&](int tile, int i) __attribute__((always_inline)) {
        const int kb = __builtin_amdgcn_readlane(ev.x, i & 63), blk = __builtin_amdgcn_readlane(ev.y, i & 63);
        pa = uniform_ptr(A + (size_t)tile * BM * row_bytes + (size_t)kb * 128);
        pw = uniform_ptr(D + (size_t)blk * 4096);
    };
    auto issue = [&](int k) __attribute__((always_inline)) {
        if (k < C::A_DMA) dma16(lds_slot + k * 1024, pa, a_voff[k]);
        else dma16(lds_slot + k * 1024, pw, w_voff[k - C::A_DMA]);
    };
    bool stored = false;   // the stores of a whole tile are behind the operands that are waited for
    // block i of tile `tile` to sum S; behind it, if there is one, the next block's operands
    auto step = [&](auto S_, int tile, int i) __attribute__((always_inline)) {
        constexpr int S = decltype(S_)::value;
        if (stored) wait_dma(2 * TT);
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        stored = false;
        uint4 fa[TT][2], fw[2][2];
        const unsigned char* ws = smem + C::A_DMA * 1024;
        if constexpr (TRANS) {
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int row = 2 * r + j;
                    fw[j][e] = *reinterpret_cast<const uint4*>(ws + row * 128 + ((4 * e + q) ^ w_row_swz(row)) * 16);
                }
        } else {
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                uint2 v[4];
#pragma unroll
                for (int x = 0; x < 4; ++x) v[x] = *reinterpret_cast<const uint2*>(ws + (16 * e + 4 * x) * 128 + lane * 8);
                fw[0][e] = make_uint4(v[0].x, v[1].x, v[2].x, v[3].x);
                fw[1][e] = make_uint4(v[0].y, v[1].y, v[2].y, v[3].y);
            }
        }
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int t = 0; t < TT; ++t) fa[t][e] = *reinterpret_cast<const uint4*>(smem + (16 * t + r) * 128 + ((4 * e + q) ^ chunk_swz<8>(r)) * 16);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        auto mma = [&](int m) __attribute__((always_inline)) {
            const int e = m / NV, t = (m % NV) >> 1, j = m & 1;
            const uint4 av = fa[t][e >> 2], bv = fw[j][e >> 2];
            const uint32_t a1 = (e & 3) == 0 ? av.x : (e & 3) == 1 ? av.y : (e & 3) == 2 ? av.z : av.w;
            const uint32_t b1 = (e & 3) == 0 ? bv.x : (e & 3) == 1 ? bv.y : (e & 3) == 2 ? bv.z : bv.w;
            acc[S][t][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(b1), __uint_as_float(a1), acc[S][t][j], 0, 0, 0);
        };
        constexpr int NMMA = 8 * NV;
        const bool last = i + 1 == n;
        // (behind the last block of all this one once more: without a branch around the products)
        const int next = !last ? i + 1 : tile + 1 < end_tile ? 0 : i, next_tile = last && tile + 1 < end_tile ? tile + 1 : tile;
        if (n > 64 && (next & 63) == 0) ev = ent[next + lane < n ? next + lane : n - 1];
        if (last && (next_tile + 1) * BM > g.M) rows_of(next_tile);
        source(next_tile, next);
#pragma unroll
        for (int m = 0, k = 0; m < NMMA; ++m) {
            // the issues spread over the first three quarters of the products
            if (k < NISSUE && m * NISSUE * 4 >= k * NMMA * 3) {
                __builtin_amdgcn_sched_barrier(0);
                issue(k);
                ++k;
                __builtin_amdgcn_sched_barrier(0);
            }
            mma(m);
        }
        __builtin_amdgcn_sched_barrier(0);
        return last;
    };

    float* const out = static_cast<float*>(g.out);
    auto store = [&](int tile) __attribute__((always_inline)) {
        const int m0 = tile * BM;
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const int row = m0 + 16 * t + r;
            f32x4 v0 = acc[0][t][0], v1 = acc[0][t][1];
#pragma unroll
            for (int s = 1; s < SUMS; ++s) {
                v0 += acc[s][t][0];
                v1 += acc[s][t][1];
            }
            float v[8];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                v[2 * i] = v0[i] + __shfl(bias, 8 * q + 2 * i, 64);
                v[2 * i + 1] = v1[i] + __shfl(bias, 8 * q + 2 * i + 1, 64);
            }
            float4* p = reinterpret_cast<float4*>(out + (size_t)row * g.N + col + 8 * q);
            if (row < g.M) {
                p[0] = make_float4(v[0], v[1], v[2], v[3]);
                p[1] = make_float4(v[4], v[5], v[6], v[7]);
            }
        }
        clear();
        stored = m0 + BM <= g.M;   // (of a tile that ends early some stores may not be there)
    };

    if (n == 0) {
        for (int tile = first; tile < end_tile; ++tile) store(tile);
        return;
    }
    source(first, 0);
#pragma unroll
    for (int k = 0; k < NISSUE; ++k) issue(k);
    for (int tile = first; tile < end_tile; ++tile) {
        for (int i = 0;; i += SUMS) {
            if (step(std::integral_constant<int, 0>{}, tile, i)) break;
            if (step(std::integral_constant<int, 1>{}, tile, i + 1)) break;
            if constexpr (SUMS == 4) {
                if (step(std::integral_constant<int, 2>{}, tile, i + 2)) break;
                if (step(std::integral_constant<int, 3>{}, tile, i + 3)) break;
            }
        }
        store(tile);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // what was asked for behind the last block still lands in this LDS
}

}  // namespace pbs
