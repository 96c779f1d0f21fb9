// dense x block-sparse -> dense (forward Y = X.W^T and input gradient dX = dY.W), one block column of the result per
// workgroup.  The smaller and sparser fp32 products (the others: pbs_split.h; of many token tiles and short columns: pbs_walk.h), and the bf16 ones whose token count or pattern gives the kernels with shared operand
// panels (pbs_dds16.h, pbs_ddsc.h) too little to share.
//
// Work decomposition.  A workgroup owns 16 TT tokens x one block column (32 columns) of the result; its KS waves take the
// column's blocks in turn (wave w blocks w, w + KS, ...) and their sums meet in LDS once, at the end.  So a launch has
// tokens / (16 TT) x columns workgroups of KS waves however few tokens or columns there are, a long column is walked KS
// times faster, and columns of any length cost what they hold: no common list of k-blocks, no step in which a wave has
// nothing to do.  TT and KS come from the cost estimate in pbs_hip.hip.  With the kernel this one replaces (tiles of 8
// columns sharing a panel, a barrier per k-block), 1 token x 4096 -> 4096 at density 0.25 took 47 us in bf16 (now 4.4),
// 101 tokens 3072 -> 768 at density 0.5 in fp32 107 us (7.2), 3072 -> 768 with Zipf rows 90 us (46), and fp32
// 4096 x 4096 x 16384 at density 0.25 1.26 ms (1.02: 134 TFLOP/s of the 155 the matrix instruction reaches in a loop).
//
// Data movement.  A wave's operands pass through LDS of its own: 16 TT x 32 dense elements and the 32 x 32 block go
// global -> LDS by DMA, are read into registers as fragments at once, and the same space takes the next block's DMA,
// which is issued one instruction at a time between the products.  No wave waits for another one before the final sum.
//   Why LDS at all: a fragment wants neighbouring lanes in neighbouring rows, and 16-byte loads whose neighbouring lanes
//   lie in different rows cost the texture path one cycle per lane (64 per instruction; a DMA instruction whose lanes
//   run along the rows takes 23 to 35).
//   Why spread: waves that issue a block's loads in one go and then its products in one go fall into step with each
//   other, so the matrix cores idle while all of them issue loads (measured: 2.38 ms for the 4096 layer instead of 1.2
//   with the loads spread, same loads, same products).
// What bounds it: fp32 the matrix cores (86 % of their rate at the large shapes; the rest is the wait and the fragment
// reads between two blocks, which three waves per SIMD hide in part); bf16 the texture path (10 KB per block and 128
// tokens at about 30 B/clk, rows of 64 bytes), small problems the chain launch -> list -> first operands (about 4 us).
//
// Matrix instructions 16x16x4 (fp32) / 16x16x32 (bf16), computed transposed: D[column][token], so a lane ends up with
// eight consecutive columns of a token and stores them with 16-byte stores, 128 (64) contiguous bytes per token.
//
// Work list ("list plan", list_plan_kernel), per pattern and direction: per block column, in order of falling block
// count, a record {column, entries, 0, 0} and the entries {k-block, data block}, by k-block, with every value inside its
// range.  Long columns are so started first.  A record has room for as many entries as there are k-blocks, so a wave asks for its first entries
// together with the number of them: one round trip to memory before the first operands instead of two (bf16 4096 -> 4096 density 0.25, 1 token
// 4.63 -> 4.39 us, 509 tokens 15.75 -> 15.49; 768 -> 3072 density 0.5, 2317 tokens, panel_kernel 14.5 -> 14.2).
#pragma once
#include "pbs_common.h"

namespace pbs {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int LIST_HEAD = 2;   // of a record's KB + 2 pairs; {column, entries} is the first
static __host__ __device__ __forceinline__ size_t list_record(int KB, int rank) { return (size_t)rank * (size_t)(KB + LIST_HEAD); }
static inline size_t list_plan_bytes(int n, int k) { return list_record(k / 32, n / 32) * 8; }

constexpr int LIST_RANK_MAX_COLS = 8192;   // ranking compares every pair of columns: beyond this, natural order

struct ListArgs {
    const int32_t *ptr, *idx;
    int nblk_n, KB, nnz;
    int* plan;
};
static inline unsigned list_plan_grid(int nblk_n) { return (unsigned)(nblk_n > 4 * 1024 ? 1024 : (nblk_n + 3) / 4); }
// One wave per column copies its entries and ranks it; workgroup `block` of `blocks` (256 threads).  Entries as the host layer keeps
// them (by k-block, every value in its range) are copied as they are; of any other list the entries outside the range and all but the first
// entry of a k-block are dropped and the rest is sorted, like in the plans of pbs_dds16.h and pbs_ddsc.h: panel_chunk_kernel goes
// through a column by k-block, and panel_kernel has room for one entry per k-block.
static __device__ __forceinline__ void list_plan(const ListArgs& a, int block, int blocks) {
    const int32_t* __restrict__ ptr = a.ptr;
    const int32_t* __restrict__ idx = a.idx;
    const int nblk_n = a.nblk_n, KB = a.KB, nnz = a.nnz;
    int* __restrict__ plan = a.plan;
    auto entry = [&](int i) { return make_int2(idx[2 * (size_t)i], idx[2 * (size_t)i + 1]); };
    auto good = [&](int2 e) { return e.x >= 0 && e.x < KB && e.y >= 0 && e.y < nnz; };
    const int lane = threadIdx.x & 63;
    for (int c = block * 4 + (threadIdx.x >> 6); c < nblk_n; c += blocks * 4) {
        const int lo = clamp_entry(ptr[c], nnz), hi = clamp_entry(ptr[c + 1], nnz);
        const int n = hi > lo ? hi - lo : 0;
        int rank = c;
        if (nblk_n <= LIST_RANK_MAX_COLS) {
            rank = 0;
            for (int o = lane; o < nblk_n; o += 64) {
                const int a = clamp_entry(ptr[o], nnz), b = clamp_entry(ptr[o + 1], nnz);
                const int m = b > a ? b - a : 0;
                rank += (m > n || (m == n && o < c)) ? 1 : 0;
            }
#pragma unroll
            for (int d = 32; d; d >>= 1) rank += __shfl_xor(rank, d, 64);
        }
        int2* const record = reinterpret_cast<int2*>(plan) + list_record(KB, rank);
        int2* const ent = record + LIST_HEAD;
        bool as_it_is = true;
#pragma unroll 4
        for (int i = lane; i < n; i += 64) {
            const int2 e = entry(lo + i);
            if (!good(e) || (i > 0 && entry(lo + i - 1).x >= e.x)) as_it_is = false;
            if (i < KB) ent[i] = make_int2(e.x < 0 ? 0 : (e.x >= KB ? KB - 1 : e.x), e.y < 0 ? 0 : (e.y >= nnz ? nnz - 1 : e.y));
        }
        int kept = n;
        if (__any(!as_it_is)) {
            // The number of the first entry of every k-block in the record's place of that k-block; then the places that have one move together.  (Lists of anything, as a
            // refused block_replace leaves them, may give every column all entries: to look for one k-block after the other took 256 columns of 100000
            // entries and 512 k-blocks 178 ms, this 1.2.)
            constexpr int NONE = 0x7fffffff;
            for (int kb = lane; kb < KB; kb += 64) __hip_atomic_store(&ent[kb].y, NONE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // (the lane that has written it above)
            __threadfence();
            for (int i = lane; i < n; i += 64) {
                const int2 e = entry(lo + i);
                if (good(e)) atomicMin(&ent[e.x].y, i);
            }
            __threadfence();
            kept = 0;
            for (int base = 0; base < KB; base += 64) {
                const int kb = base + lane;
                const int first = kb < KB ? __hip_atomic_load(&ent[kb].y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : NONE;
                const unsigned long long there = __ballot(first != NONE);
                if (first != NONE) ent[kept + __popcll(there & ((1ull << lane) - 1))] = make_int2(kb, entry(lo + first).y);   // (places of this round and before)
                kept += __popcll(there);
            }
        }
        if (lane < LIST_HEAD) record[lane] = lane == 0 ? make_int2(c, kept) : make_int2(0, 0);
    }
}
__global__ __launch_bounds__(256) void list_plan_kernel(ListArgs a) { list_plan(a, blockIdx.x, gridDim.x); }

struct StreamArgs {
    const void* a;      // [M, K] row-major
    const void* data;   // [nnz*32, 32]
    const int* plan;    // the list plan
    const void* bias;   // nullptr or [N]
    void* out;          // [M, N] row-major
    int M, N, K;
    int m_tiles;
    int xcd_t;          // the XCDs are xcd_t ranges of token tiles x 8 / xcd_t sets of columns
    int group;          // token tiles that share one pass over the columns
};

// TRANS = 0: B[k][n] = block[k*32 + n]   (forward: the packed block is W_block^T = [in][out])
// TRANS = 1: B[k][n] = block[n*32 + k]   (dX: contraction runs along the packed block's rows)
template <typename T, int TRANS, int TT, int KS>
struct StreamCfg {
    using E = Elem<T>;
    static constexpr int BM = 16 * TT;
    static constexpr int ROWB = 32 * E::ESZ;               // bytes of a row of a k-block
    static constexpr int CPR = ROWB / 16;
    static constexpr int RPI = 64 / CPR;                   // rows of one DMA instruction
    static constexpr int A_DMA = BM / RPI;
    static constexpr int W_DMA = 32 / RPI;
    static constexpr int SLOT = (A_DMA + W_DMA) * 1024;
    static constexpr int RED = KS * 2 * TT * 64 * 16;
    static constexpr int LDS = KS * SLOT > RED ? KS * SLOT : RED;
};

// Chunk c (16 bytes) of panel row r sits at place c ^ chunk_swz(r): the lanes' reads of one chunk of 16 rows then touch
// every LDS bank once.  bf16 rows have 4 chunks, fp32 rows 8.
template <int CPR>
static __device__ __forceinline__ int chunk_swz(int r) {
    return CPR == 4 ? ((r >> 2) & 3) : ((r >> 1) & 7);
}

template <typename T, int TRANS, int TT, int KS, int WPE>
__global__ __launch_bounds__(KS * 64, WPE) void stream_kernel(StreamArgs g) {
    using C = StreamCfg<T, TRANS, TT, KS>;
    using E = Elem<T>;
    constexpr int BM = C::BM, ESZ = E::ESZ, NV = 2 * TT, CPR = C::CPR;
    constexpr int NI = ESZ == 4 ? 2 : 1;                   // 16-byte pieces of k per lane
    __shared__ __attribute__((aligned(1024))) unsigned char smem[C::LDS];

    const int ncols = g.N >> 5;
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
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4;

    // this wave's entries are wave, wave + KS, ...: its next 64, one per lane, and with the first of them the number of all
    const int2* const record = reinterpret_cast<const int2*>(g.plan) + list_record(g.K >> 5, cr);
    const int2* const ent = record + LIST_HEAD + wave;
    const int room = ((g.K >> 5) - 1 - wave) / KS;   // (a record's last place for an entry of this wave's; of a wave behind the last k-block 0, and not read)
    int2 ev = make_int2(0, 0);
    if (wave < g.K >> 5) ev = ent[(size_t)(lane < room ? lane : room) * KS];
    const int2 head = record[0];
    const int n = head.y;
    const int col = head.x * 32;

    const unsigned char* A = static_cast<const unsigned char*>(g.a) + (size_t)m0 * g.K * ESZ;
    const unsigned char* D = static_cast<const unsigned char*>(g.data);
    unsigned char* slot = smem + wave * C::SLOT;
    const unsigned lds_slot = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)slot);

    unsigned a_voff[C::A_DMA];
#pragma unroll
    for (int i = 0; i < C::A_DMA; ++i) {
        int row = i * C::RPI + lane / CPR;
        const int chunk = (lane % CPR) ^ chunk_swz<CPR>(row);
        if (m0 + row >= g.M) row = g.M - 1 - m0;
        a_voff[i] = (unsigned)row * (unsigned)(g.K * ESZ) + chunk * 16;
    }
    // The block.  TRANS ([n][k] as stored): rows swizzled so that the lanes' 16-byte reads of 16 rows meet no bank twice.
    // Else ([k][n]): fp32 rows are put in the order (k / 16, k % 4, k / 4 % 4), which makes every read linear in the lane;
    // bf16 stays as stored, for the transposing reads.
    auto w_row_swz = [](int row) { return ESZ == 4 ? ((row >> 1) & 7) : ((row >> 3) & 3); };
    unsigned w_voff[C::W_DMA];
#pragma unroll
    for (int i = 0; i < C::W_DMA; ++i) {
        if constexpr (TRANS) {
            const int row = i * C::RPI + lane / CPR;
            w_voff[i] = row * C::ROWB + ((lane % CPR) ^ w_row_swz(row)) * 16;
        } else if constexpr (ESZ == 4) {
            const int p = i * 8 + lane / 8;
            w_voff[i] = ((p & 16) + 4 * (p & 3) + ((p >> 2) & 3)) * 128 + (lane & 7) * 16;
        } else {
            w_voff[i] = i * 1024 + lane * 16;
        }
    }

    f32x4 acc[TT][2];
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[t][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    if (wave < n) {
        const int mine = (n - wave + KS - 1) / KS;   // entries wave, wave + KS, ...
        auto a_src = [&](int2 e) { return uniform_ptr(A + (size_t)e.x * C::ROWB); };
        auto w_src = [&](int2 e) { return uniform_ptr(D + (size_t)e.y * (1024 * ESZ)); };
        constexpr int NISSUE = C::A_DMA + C::W_DMA;
        auto issue = [&](int k, const unsigned char* pa, const unsigned char* pw) __attribute__((always_inline)) {
            if (k < C::A_DMA) dma16(lds_slot + k * 1024, pa, a_voff[k]);
            else dma16(lds_slot + k * 1024, pw, w_voff[k - C::A_DMA]);
        };
        uint4 fa[TT][NI], fw[2][NI];
        // column of the result that row rho of parity j stands for: fp32 2 rho + j, bf16 8 (rho / 4) + 4 j + rho % 4; either
        // way a lane ends up with the eight columns 8 q .. 8 q + 7
        auto read_frags = [&]() __attribute__((always_inline)) {
            const unsigned char* ws = slot + C::A_DMA * 1024;
            if constexpr (TRANS) {
#pragma unroll
                for (int i = 0; i < NI; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const int row = ESZ == 4 ? 2 * r + j : 8 * (r >> 2) + 4 * j + (r & 3);
                        fw[j][i] = *reinterpret_cast<const uint4*>(ws + row * C::ROWB + ((4 * i + q) ^ w_row_swz(row)) * 16);
                    }
            } else if constexpr (ESZ == 4) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    uint2 v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = *reinterpret_cast<const uint2*>(ws + (16 * i + 4 * e) * 128 + lane * 8);
                    fw[0][i] = make_uint4(v[0].x, v[1].x, v[2].x, v[3].x);
                    fw[1][i] = make_uint4(v[0].y, v[1].y, v[2].y, v[3].y);
                }
            } else {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const unsigned char* p = ws + (8 * q + (r >> 2)) * 64 + (r & 3) * 16 + 8 * j;
                    const uint2 lo = tr16_b64(p), hi = tr16_b64(p + 256);
                    fw[j][0] = make_uint4(lo.x, lo.y, hi.x, hi.y);
                }
            }
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int t = 0; t < TT; ++t)
                    fa[t][i] = *reinterpret_cast<const uint4*>(slot + (16 * t + r) * C::ROWB + ((4 * i + q) ^ chunk_swz<CPR>(r)) * 16);
        };
        constexpr int NSTEP = ESZ == 4 ? 8 : 1;            // matrix instructions per accumulator and block
        constexpr int NMMA = NSTEP * NV;
        auto mma1 = [&](int m) __attribute__((always_inline)) {
            const int s = m / NV, t = (m % NV) >> 1, j = m & 1;
            if constexpr (ESZ == 4) {
                const uint4 a = fa[t][s >> 2], b = fw[j][s >> 2];
                const int e = s & 3;
                const uint32_t av = e == 0 ? a.x : e == 1 ? a.y : e == 2 ? a.z : a.w;
                const uint32_t bv = e == 0 ? b.x : e == 1 ? b.y : e == 2 ? b.z : b.w;
                acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(bv), __uint_as_float(av), acc[t][j], 0, 0, 0);
            } else {
                acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, fw[j][0]), __builtin_bit_cast(bf16x8, fa[t][0]),
                                                                    acc[t][j], 0, 0, 0);
            }
        };

        auto entry = [&](int i) __attribute__((always_inline)) {
            return make_int2(__builtin_amdgcn_readlane(ev.x, i & 63), __builtin_amdgcn_readlane(ev.y, i & 63));
        };
        int2 e1 = entry(0);
        {
            const unsigned char* pa = a_src(e1);
            const unsigned char* pw = w_src(e1);
#pragma unroll
            for (int k = 0; k < NISSUE; ++k) issue(k, pa, pw);
        }
        // one block: its operands have been on their way since the block before; the next one's are asked for between the products
        auto step = [&](bool more) __attribute__((always_inline)) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            read_frags();
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            if (more) {
                const unsigned char* pa = a_src(e1);
                const unsigned char* pw = w_src(e1);
#pragma unroll
                for (int m = 0, k = 0; m < NMMA; ++m) {
                    // the issues spread over the first three quarters of the products
                    if (k < NISSUE && m * NISSUE * 4 >= k * NMMA * 3) {
                        __builtin_amdgcn_sched_barrier(0);
                        issue(k, pa, pw);
                        ++k;
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    mma1(m);
                    if (m == NMMA - 1)
                        for (; k < NISSUE; ++k) issue(k, pa, pw);
                }
            } else {
#pragma unroll
                for (int m = 0; m < NMMA; ++m) mma1(m);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        for (int i = 0; i + 1 < mine; ++i) {
            if (((i + 1) & 63) == 0) {
                const int l = i + 1 + lane;
                ev = ent[(size_t)(l < mine ? l : mine - 1) * KS];
            }
            e1 = entry(i + 1);
            step(true);
        }
        step(false);
    }

    T* out = static_cast<T*>(g.out);
    const T* bias = static_cast<const T*>(g.bias);
    // a lane's eight results of a token: columns 8 q .. 8 q + 7 (register i of parity j is column 8 q + 2 i + j)
    auto store = [&](int t, const f32x4& v0, const f32x4& v1) __attribute__((always_inline)) {
        const int row = m0 + 16 * t + r;
        if (row >= g.M) return;
        float v[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            v[ESZ == 4 ? 2 * i : i] = v0[i];
            v[ESZ == 4 ? 2 * i + 1 : i + 4] = v1[i];
        }
        if (bias) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] += E::to_f32(bias[col + 8 * q + i]);
        }
        T* p = out + (size_t)row * g.N + col + 8 * q;
        if constexpr (ESZ == 4) {
            reinterpret_cast<float4*>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
            reinterpret_cast<float4*>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
        } else {
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                w[i] = (uint32_t)E::from_f32(v[2 * i]).bits | ((uint32_t)E::from_f32(v[2 * i + 1]).bits << 16);
            *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    };
    if constexpr (KS == 1) {
#pragma unroll
        for (int t = 0; t < TT; ++t) store(t, acc[t][0], acc[t][1]);
    } else {
        f32x4* red = reinterpret_cast<f32x4*>(smem);
        __syncthreads();   // the slots are reused
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int j = 0; j < 2; ++j) red[(wave * NV + 2 * t + j) * 64 + lane] = acc[t][j];
        __syncthreads();
        for (int t = wave; t < TT; t += KS) {
            f32x4 v0 = red[(2 * t) * 64 + lane], v1 = red[(2 * t + 1) * 64 + lane];
#pragma unroll
            for (int w = 1; w < KS; ++w) {
                v0 += red[(w * NV + 2 * t) * 64 + lane];
                v1 += red[(w * NV + 2 * t + 1) * 64 + lane];
            }
            store(t, v0, v1);
        }
    }
}

}  // namespace pbs
