// Weight gradient in fp32 on the bf16 matrix cores: the units of pbs_sdd_row.h (up to four blocks of a block row over a slice of the
// tokens, each of four waves every fourth chunk of 32 tokens), with every value in three bfloat16 parts and six of their nine products, as in
// pbs_split.h (range and what does not fit: see there; a block whose sum is not finite is computed again with fp32 instructions).
//
// A chunk's twelve products of a block (two halves of 16 tokens) are summed by themselves, small ones first, and then added to the block's total,
// so the error against 64 bits does not grow with the length of a wave's share.
//
// What bounds it: vector instructions.  A chunk of four blocks is 4 x 384 cycles of matrix instructions (4 x 1024 with fp32 ones) and 5 pieces x 104
// instructions that split, so a wave's vector instructions run between its matrix instructions: while one half of a block is
// multiplied, the other half, or the first half of the next block, is split into the registers that the half before has left.  The pieces pass
// through the wave's own LDS as in pbs_sdd_row.h: read 4 bytes at a time, the lane's feature of the tokens 2 e + h, so that both
// operands have the tokens of a half in one order.
#pragma once
#include "pbs_common.h"
#include "pbs_sdd_row.h"
#include "pbs_split.h"

namespace pbs {

typedef unsigned u32x4v __attribute__((ext_vector_type(4)));

// a half of a piece: 8 tokens of one feature, and its parts
struct HalfRaw {
    float v[8];
    // half kk of the piece in LDS: tokens 16 kk + 2 e + h
    __device__ __forceinline__ void read(const unsigned char* piece, int kk, int lane) {
        const unsigned char* p = piece + kk * 2048 + (lane >> 5) * 128 + (lane & 31) * 4;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = *reinterpret_cast<const float*>(p + e * 256);
    }
    __device__ __forceinline__ float sum() const { return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])); }
};
struct HalfParts {
    uint32_t w[3][4];
    __device__ __forceinline__ void split(const HalfRaw& r, int i, float scale = SP_SCALE) {   // values 2 i and 2 i + 1
        split2(r.v[2 * i] * scale, r.v[2 * i + 1] * scale, w[0][i], w[1][i], w[2][i]);
    }
    __device__ __forceinline__ bf16x8 part(int p) const { return __builtin_bit_cast(bf16x8, u32x4v{w[p][0], w[p][1], w[p][2], w[p][3]}); }
};
// The products of a chunk and block, in this order: five small ones of the first half (`first`: into a new sum), five of the second half, and on
// top of them the two large ones.  The matrix instruction cuts what is far below its largest term off towards minus infinity: a chunk's sum is
// a fifteenth of a unit in the last place too low on average, and the sum of many has a mean error that grows with their number (-1.4e-7 of the
// results' size at 16384 tokens).  So every other chunk is made with G's sign changed and subtracted.
static __device__ __forceinline__ void mma_parts(f32x16& c, bf16x8 g, bf16x8 x) { c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(g, x, c, 0, 0, 0); }
static __device__ __forceinline__ void small_mma(f32x16& c, const HalfParts& g, const HalfParts& x, int m, bool first) {
    constexpr int PG[5] = {2, 1, 0, 1, 0}, PX[5] = {0, 1, 2, 0, 1};
    if (first && m == 0) {
#pragma unroll
        for (int v = 0; v < 16; ++v) c[v] = 0.f;
    }
    mma_parts(c, g.part(PG[m]), x.part(PX[m]));
}

// Chunks c_lo .. c_hi - 1 of a unit of NB blocks.
template <int NB>
static __device__ __forceinline__ void sdd_split_body(const SddRowArgs& a, const int* __restrict__ unit, int c_lo, int c_hi, float* partial,
                                                      unsigned char* smem, int lane, int wave) {
    using C = SddRowCfg<float>;
    constexpr int PIECE = C::PIECE, GS = NB <= 2 ? 2 : 1, XS = ROW_PIECES - GS;
    const int r = lane & 31, h = lane >> 5;
    const int row = unit[0];
    int cblk[NB], bblk[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        cblk[b] = unit[4 + b];
        bblk[b] = unit[4 + ROW_SIZES + b];
    }
    const bool sums = a.bias_out && unit[2] == 0;

    const size_t gs = (size_t)a.N * 4, xs = (size_t)a.K * 4;   // row strides
    const unsigned char* G = static_cast<const unsigned char*>(a.g) + (size_t)row * 128;
    const unsigned char* X = static_cast<const unsigned char*>(a.x);
    unsigned char* mem = smem + wave * C::WAVE_LDS;   // GS pieces of G, XS of X
    const unsigned lds = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)mem);
    RowSource<false, 4, 8> from_g(G, gs, a.M, lane / 8, lane % 8), from_x(X, xs, a.M, lane / 8, lane % 8);
    auto dma_g = [&](int slot, int chunk, int i) __attribute__((always_inline)) {
        from_g.dma(lds + slot * PIECE + i * 1024, chunk, 0, i);
    };
    auto dma_x = [&](int slot, int chunk, int c, int i) __attribute__((always_inline)) {
        from_x.dma(lds + (GS + slot) * PIECE + i * 1024, chunk, c * 128, i);
    };

    f32x16 total[NB], part[2];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) total[b][v] = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) part[0][v] = part[1][v] = 0.f;
    float bsum = 0.f, bleft = 0.f;

    int chunk = c_lo + wave;
    if (chunk < c_hi) {
        const int last = chunk + (c_hi - 1 - chunk) / ROW_NW * ROW_NW;   // this wave's last chunk
        auto after = [&](int c, int n) { return c + n * ROW_NW <= last ? c + n * ROW_NW : last; };   // (past the end: the last one again)
        // X piece q is block q % NB of this wave's chunk q / NB, in slot q % XS
#pragma unroll
        for (int t = 0; t < GS; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) dma_g(t, after(chunk, t), i);
#pragma unroll
        for (int q = 0; q < XS; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) dma_x(q, after(chunk, q / NB), cblk[q % NB], i);
        wait_dma((XS - 1) * 4);
        auto sign_of = [](int c) { return (c ^ (c >> 2)) & 1 ? -1.f : 1.f; };   // (a wave has every fourth chunk: it and its neighbours alternate)
        HalfRaw gr[2], xr[2];
        HalfParts gp[2], xp[2];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            gr[kk].read(mem, kk, lane);
            xr[kk].read(mem + GS * PIECE, kk, lane);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            gp[0].split(gr[0], i, SP_SCALE * sign_of(chunk));
            xp[0].split(xr[0], i);
        }
        float sign = sign_of(chunk), sign_before = 1.f;
        int xat = 0, gat = 0;   // slots of the pieces that have been read last
        int early = (XS - 1 + NB - 1) / NB;   // chunks: the pieces asked for above have fewer DMA instructions behind them than the later ones
        for (;; chunk += ROW_NW) {
            if (sums) add_with_rest(bsum, bleft, gr[0].sum() + gr[1].sum());
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const int xnext = xat + 1 == XS ? 0 : xat + 1, gnext = GS == 2 ? gat ^ 1 : 0;
                const bool end = b == NB - 1;
                f32x16& c = part[b & 1];
                // -- first half: its parts are there; the second half's are made --
                // X piece q + 1 has been asked for XS - 1 blocks ago: behind it there are the pieces up to q - 1 + XS and, where a
                // chunk began in between, a G piece
                constexpr auto younger = [](int b) constexpr {
                    int n = (XS - 2) * 4;
                    for (int d = 2; d <= XS; ++d)
                        if (((b + 1 - d) % NB + NB) % NB == 0) n += 4;
                    return n;
                };
                constexpr int YG = GS == 1 ? (NB - 2) * 4 : (2 * NB - 2) * 4 + (NB >= 2 ? 4 : 0);
                const int y = early > 0 ? (XS - 2) * 4 : younger(b);
                wait_dma(end && YG < y ? YG : y);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int m = 0; m < 5; ++m) {
                    small_mma(c, gp[0], xp[0], m, true);
                    if (m < 4) {
                        xp[1].split(xr[1], m);
                        if (b == 0) gp[1].split(gr[1], m, SP_SCALE * sign);
                    }
                    if (m == 4) {
                        xr[0].read(mem + (GS + xnext) * PIECE, 0, lane);
                        if (end) gr[0].read(mem + gnext * PIECE, 0, lane);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                // -- second half; the next block's first half is split, the block before joins its total --
                const bf16x8 g_large = gp[0].part(0), x_large = xp[0].part(0);
#pragma unroll
                for (int m = 0; m < 7; ++m) {
                    if (m < 5) small_mma(c, gp[1], xp[1], m, false);
                    else if (m == 5) mma_parts(c, g_large, x_large);
                    else mma_parts(c, gp[1].part(0), xp[1].part(0));
                    if (m < 4) {
                        xp[0].split(xr[0], m);
                        if (end) gp[0].split(gr[0], m, SP_SCALE * sign_of(chunk + ROW_NW));
                        // this block's slot (and at the start of a chunk G's) has been read: the splits above have waited for that
                        dma_x(xat, after(chunk, (b + XS) / NB), cblk[(b + XS) % NB], m);
                    } else if (b == 0 && m < 6) {
                        dma_g(gat, after(chunk, GS), 2 * (m - 4));
                        dma_g(gat, after(chunk, GS), 2 * (m - 4) + 1);
                    }
                    if (m == 4) {
                        xr[1].read(mem + (GS + xnext) * PIECE, 1, lane);
                        if (end) gr[1].read(mem + gnext * PIECE, 1, lane);
                    }
                    if (m < 4) {
#pragma unroll
                        for (int v = 4 * m; v < 4 * m + 4; ++v)
                            total[(b + NB - 1) % NB][v] = __builtin_fmaf(part[(b & 1) ^ 1][v], b == 0 ? sign_before : sign, total[(b + NB - 1) % NB][v]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (NB % 2 == 1) {
                    // (an odd number of blocks: the last one's sums move to where the first block of the next chunk looks for them)
                    if (end) {
                        const f32x16 t = part[0];
                        part[0] = part[1];
                        part[1] = t;
                    }
                }
                xat = xnext;
                if (end) gat = gnext;
            }
            --early;
            sign_before = sign;
            sign = sign_of(chunk + ROW_NW);
            if (chunk >= last) break;
        }
        // the last block of the last chunk
#pragma unroll
        for (int v = 0; v < 16; ++v) total[NB - 1][v] = __builtin_fmaf(part[1][v], sign_before, total[NB - 1][v]);
        wait_dma(0);   // the sums below use the same space
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }

    // ---- the waves' sums meet in LDS, two blocks at a time: wave 2 k + jj stores columns 16 jj .. + 15 of block k ----
    f32x4* red = reinterpret_cast<f32x4*>(smem);
#pragma unroll
    for (int b0 = 0; b0 < NB; b0 += 2) {
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 2; ++k)
            if (b0 + k < NB)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const f32x16& t = total[(b0 + k) % NB];
                    red[((wave * 2 + k) * 4 + i) * 64 + lane] = f32x4{t[4 * i], t[4 * i + 1], t[4 * i + 2], t[4 * i + 3]};
                }
        __syncthreads();
        const int k = wave >> 1, jj = wave & 1;
        const int at = k == 0 ? bblk[b0] : bblk[(b0 + 1) % NB];
        if (b0 + k < NB && at >= 0) {
            f32x4 v[2];   // quad q = 2 jj + i: columns 8 q + 4 h .. + 3 of row r
            float off = 0.f;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                v[i] = red[(k * 4 + 2 * jj + i) * 64 + lane];
#pragma unroll
                for (int w = 1; w < ROW_NW; ++w) v[i] += red[((w * 2 + k) * 4 + 2 * jj + i) * 64 + lane];
                v[i] *= SP_UNSCALE;
#pragma unroll
                for (int e = 0; e < 4; ++e) off = __builtin_fmaf(v[i][e], 0.f, off);
            }
            if (__any(off != 0.f)) {
                // again, with fp32 instructions: infinities, NaN, sums beyond the scaled range.  A chunk's products by themselves, then what would be a
                // wave's chunks, as in pbs_sdd_row.h.
                f32x16 sum;
#pragma unroll
                for (int e = 0; e < 16; ++e) sum[e] = 0.f;
                const float* g = static_cast<const float*>(a.g) + row * 32 + r;
                const float* x = static_cast<const float*>(a.x) + (k == 0 ? cblk[b0] : cblk[(b0 + 1) % NB]) * 32 + r;
#pragma unroll 1
                for (int w = 0; w < ROW_NW; ++w) {
                    f32x16 of_wave;
#pragma unroll
                    for (int e = 0; e < 16; ++e) of_wave[e] = 0.f;
#pragma unroll 1
                    for (int c = c_lo + w; c < c_hi && c * ROW_TC < a.M; c += ROW_NW) {
                        f32x16 s;
#pragma unroll
                        for (int e = 0; e < 16; ++e) s[e] = 0.f;
#pragma unroll 1
                        for (int t0 = c * ROW_TC; t0 < (c + 1) * ROW_TC; t0 += 16) {
                            float gk[8], xk[8];
#pragma unroll
                            for (int e = 0; e < 8; ++e) {
                                const int t = t0 + 2 * e + h, at = t < a.M ? t : a.M - 1;
                                gk[e] = g[(size_t)at * a.N];
                                xk[e] = x[(size_t)at * a.K];
                                if (t >= a.M) gk[e] = xk[e] = 0.f;
                            }
#pragma unroll
                            for (int e = 0; e < 8; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(gk[e], xk[e], s, 0, 0, 0);
                        }
                        of_wave += s;
                    }
                    sum += of_wave;
                }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (v[i][e] - v[i][e] != 0.f) v[i][e] = jj == 0 ? sum[4 * i + e] : sum[8 + 4 * i + e];
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                float* p = (partial ? partial : static_cast<float*>(a.out)) + (size_t)at * 1024 + r * 32 + 8 * (2 * jj + i) + 4 * h;
                if (a.add) v[i] += *reinterpret_cast<const f32x4*>(p);
                *reinterpret_cast<f32x4*>(p) = v[i];
            }
        }
    }
    if (sums) {
        float* s = reinterpret_cast<float*>(smem + ROW_NW * 2 * 4 * 1024);
        bsum += __shfl_xor(bsum, 32, 64);
        if (lane < 32) s[wave * 32 + lane] = bsum;
        __syncthreads();
        if (wave == 0 && lane < 32) {
            float v = s[lane];
#pragma unroll
            for (int w = 1; w < ROW_NW; ++w) v += s[w * 32 + lane];
            float* p = (partial ? partial + (size_t)a.nnz * 1024 : static_cast<float*>(a.bias_out)) + row * 32 + lane;
            *p = a.add ? *p + v : v;
        }
    }
}

// (workgroups and units as in sdd_row_kernel)
__global__ __launch_bounds__(ROW_NW * 64, SddRowCfg<float>::WPE) void sdd_split_kernel(SddRowArgs a) {
    __shared__ __attribute__((aligned(1024))) unsigned char smem[SddRowCfg<float>::LDS];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    RowTask t;
    if (!row_task(a, t)) return;
    switch (t.unit[1]) {
        case 4: sdd_split_body<4>(a, t.unit, t.c_lo, t.c_hi, t.partial, smem, lane, wave); break;
        case 3: sdd_split_body<3>(a, t.unit, t.c_lo, t.c_hi, t.partial, smem, lane, wave); break;
        case 2: sdd_split_body<2>(a, t.unit, t.c_lo, t.c_hi, t.partial, smem, lane, wave); break;
        case 1: sdd_split_body<1>(a, t.unit, t.c_lo, t.c_hi, t.partial, smem, lane, wave); break;
        default:
            if (a.bias_out) sdd_row_body<float, 0, false>(a, t.unit, t.c_lo, t.c_hi, t.partial, smem, lane, wave);
            break;
    }
}

}  // namespace pbs
