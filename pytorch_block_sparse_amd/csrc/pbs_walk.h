// dense x block-sparse -> dense in fp32 for many token tiles and short columns: one wave per block column and tile of 32 tokens.
//
// stream_kernel (pbs_stream.h) starts a workgroup of two waves per token tile and column: list, first operands, a few blocks each, the sum of the two in LDS behind two barriers,
// the stores.  Here a wave takes its column alone: there is nothing to share and no barrier, the four waves of a SIMD are at different places of theirs, and a column of three
// blocks is not two blocks' time long.  The column's blocks go to two sums in turn, which are added like those of stream_kernel's waves: a token's result has the same bits as there.
//
// What bounds it: the texture path (8 KB per block, 0.87 of the cycles of its matrix instructions) and memory.  Tiles of 64 tokens copy 12 KB for twice the
// products, but 12 KB and 162 registers a wave leave three waves to a SIMD: 2 to 20 % slower; of 48 tokens between the two, of 16 5 to 15 % slower, of 128 spilled.
// Measured, us, stream_kernel -> here: 672 -> 3200 density 0.21, 3133 tokens 39.1 -> 31.1; 352 -> 2080 density 0.15, 8586 tokens 33.8 -> 29.3; 704 -> 1856 density 0.09, 8054 tokens
// 32.1 -> 27.9; 992 -> 1984 density 0.25 with Zipf rows, 4001 tokens 48.8 -> 43.0; 448 -> 640 density 0.46, 14976 tokens 44.0 -> 39.7.
#pragma once
#include <type_traits>

#include "pbs_common.h"
#include "pbs_stream.h"

namespace pbs {

constexpr int WALK_TT = 2;         // token tile in units of 16
constexpr int WALK_MAX_K = 1024;   // (a lane for every entry of a column's list; why not more: choose_walk)

// TRANS as in stream_kernel, whose launch of two waves in tiles of WALK_TT this one's workgroups stand for.
template <int TRANS>
__global__ __launch_bounds__(64, 4) void walk_kernel(StreamArgs g) {
    using C = StreamCfg<float, TRANS, WALK_TT, 1>;
    constexpr int TT = WALK_TT, BM = C::BM, NV = 2 * TT;
    static_assert(WALK_MAX_K <= 64 * 32, "the whole list in one register pair");
    __shared__ __attribute__((aligned(1024))) unsigned char smem[C::SLOT];

    const int ncols = g.N >> 5, KB = g.K >> 5;
    const int xcd = blockIdx.x % NUM_XCD, local = blockIdx.x / NUM_XCD;
    const int xt = xcd % g.xcd_t, xc = xcd / g.xcd_t, cstep = NUM_XCD / g.xcd_t;
    // this XCD: token tiles t_lo .. t_hi - 1, ranked columns xc, xc + cstep, ...
    const int t_lo = (int)((long long)g.m_tiles * xt / g.xcd_t), t_hi = (int)((long long)g.m_tiles * (xt + 1) / g.xcd_t);
    const int nc = (ncols - xc + cstep - 1) / cstep;
    if (local >= (t_hi - t_lo) * nc) return;
    const int gsz = g.group * nc;
    const int grp = local / gsz, rem = local - grp * gsz;
    int tg = t_hi - t_lo - grp * g.group;
    tg = tg < g.group ? tg : g.group;
    const int ci = rem / tg;
    const int cr = xc + ci * cstep;
    const int m0 = (t_lo + grp * g.group + rem - ci * tg) * BM;

    const int lane = threadIdx.x & 63;
    const int r = lane & 15, q = lane >> 4;
    const int2* const record = reinterpret_cast<const int2*>(g.plan) + list_record(KB, cr);
    const int2 ev = record[LIST_HEAD + (lane < KB ? lane : KB - 1)];
    const int2 head = record[0];
    const int n = __builtin_amdgcn_readfirstlane(head.y);
    const int col = __builtin_amdgcn_readfirstlane(head.x) * 32;
    const float bias = g.bias ? static_cast<const float*>(g.bias)[col + (lane & 31)] : 0.f;   // of column lane % 32

    const unsigned row_bytes = (unsigned)g.K * 4u;
    const unsigned char* const A = static_cast<const unsigned char*>(g.a) + (size_t)m0 * row_bytes;
    const unsigned char* const D = static_cast<const unsigned char*>(g.data);
    const unsigned lds_slot = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)smem);

    unsigned a_voff[C::A_DMA];
#pragma unroll
    for (int i = 0; i < C::A_DMA; ++i) {   // (tokens behind the last one re-read that)
        const int row = i * C::RPI + lane / 8, chunk = (lane & 7) ^ chunk_swz<8>(row), left = g.M - 1 - m0;
        a_voff[i] = (unsigned)(row < left ? row : left) * row_bytes + chunk * 16;
    }
    auto w_row_swz = [](int row) { return (row >> 1) & 7; };
    unsigned w_voff[C::W_DMA];
#pragma unroll
    for (int i = 0; i < C::W_DMA; ++i) {
        const int row = i * 8 + lane / 8;
        if constexpr (TRANS) w_voff[i] = row * 128 + ((lane & 7) ^ w_row_swz(row)) * 16;
        else w_voff[i] = ((row & 16) + 4 * (row & 3) + ((row >> 2) & 3)) * 128 + (lane & 7) * 16;
    }

    f32x4 acc[2][TT][2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[s][t][0] = acc[s][t][1] = f32x4{0.f, 0.f, 0.f, 0.f};

    constexpr int NISSUE = C::A_DMA + C::W_DMA;
    const unsigned char *pa = nullptr, *pw = nullptr;   // the operands being asked for
    auto source = [&](int i) __attribute__((always_inline)) {
        pa = uniform_ptr(A + (size_t)__builtin_amdgcn_readlane(ev.x, i) * 128);
        pw = uniform_ptr(D + (size_t)__builtin_amdgcn_readlane(ev.y, i) * 4096);
    };
    auto issue = [&](int k) __attribute__((always_inline)) {
        if (k < C::A_DMA) dma16(lds_slot + k * 1024, pa, a_voff[k]);
        else dma16(lds_slot + k * 1024, pw, w_voff[k - C::A_DMA]);
    };
    // block i to sum S; between its products the next block's operands are asked for
    auto step = [&](auto S_, int i) __attribute__((always_inline)) {
        constexpr int S = decltype(S_)::value;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
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
        source(i + 1 < n ? i + 1 : i);   // (behind the last block that once more: a branch around the products and a second copy of them cost 1 to 10 %)
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
    };
    if (n > 0) {
        source(0);
#pragma unroll
        for (int k = 0; k < NISSUE; ++k) issue(k);
        for (int i = 0; i < n; i += 2) {
            step(std::integral_constant<int, 0>{}, i);
            if (i + 1 < n) step(std::integral_constant<int, 1>{}, i + 1);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (what was asked for behind the last block still lands in this LDS)

#pragma unroll
    for (int t = 0; t < TT; ++t) {
        const int row = m0 + 16 * t + r;
        const f32x4 v0 = acc[0][t][0] + acc[1][t][0], v1 = acc[0][t][1] + acc[1][t][1];
        float v[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[2 * i] = v0[i] + __shfl(bias, 8 * q + 2 * i, 64);
            v[2 * i + 1] = v1[i] + __shfl(bias, 8 * q + 2 * i + 1, 64);
        }
        float4* p = reinterpret_cast<float4*>(static_cast<float*>(g.out) + (size_t)row * g.N + col + 8 * q);
        if (row < g.M) {
            p[0] = make_float4(v[0], v[1], v[2], v[3]);
            p[1] = make_float4(v[4], v[5], v[6], v[7]);
        }
    }
}

}  // namespace pbs
