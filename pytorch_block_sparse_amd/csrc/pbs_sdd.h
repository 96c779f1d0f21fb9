// What the two kernels of dense^T x dense -> block-sparse (weight gradient on the sparse support) share:
//   out[32b + j][i] = sum_t G[t][32r + i] * X[t][32c + j]   for every data block b at (r, c).
// With more than one token slice the fp32 partial blocks go to a workspace and sdd_reduce_kernel adds them in slice order,
// so that the result does not depend on scheduling.  Also the choice of rows of a rectangle for pbs_sdd_bf16.h.
#pragma once
#include "pbs_common.h"

namespace pbs {

struct SddArgs {
    const void* g;           // [M, N] grad_output, row-major
    const void* x;           // [M, K] input, row-major
    const int32_t* ptr;      // row_start_ends_a [N/32 + 1]
    const int32_t* idx;      // cols_a [nnz][2] = (block col, data block)
    void* out;               // [nnz*32, 32] (T) when nsplit == 1
    void* bias_out;          // nullptr or [N] (T)
    float* partial;          // [nsplit][nnz*1024, then N] fp32 when nsplit > 1
    int M, N, K, nnz;
    int rows;                // block rows of a rectangle, 16 or 8
    int even;                // whether the rows are spread evenly over the bands
    int band_room;           // then: blocks of a band that its rectangles hold in as many passes as the average one takes
    int tiles_r, tiles_c, nsplit;
    int tokens_per_split;    // multiple of TC
};

// Which block rows of W form row band `band` of rectangles (SR places; -1 = no row).  Normally they are
// rows SR*band .. SR*band + SR - 1, or (`even`) as many consecutive ones as in the other bands.  When the per-row block counts are very uneven (largest > 2x the
// mean) the rows are ranked by count and dealt to the bands in serpentine order, so that all
// rectangles hold about the same number of blocks.  So they are in an even partition, which is there for rectangles that take one pass less over their tokens, when
// the fullest band has more than `band_room` blocks, with which its rectangles take a pass more than the average one: where long rows
// are full the largest is below twice the mean and bands as uneven as they get.  (300 problems with Zipf rows in even partitions: without it 1.12 times as fast as in as few rectangles as
// possible, 88 of them slower, down to 0.73; with it 1.24 times, 20 slower, down to 0.81.  2304 -> 2848 density 0.63, 8606 tokens 199 -> 124 us.  Without structure one in a hundred is dealt: level.)
// Every workgroup derives its own band from the
// row pointer array (a few microseconds at most; above SDD_BALANCE_MAX_ROWS rows the natural order
// is kept).  Called by all threads of the workgroup; `scratch` is LDS for nblk_r ints.  Returns
// whether the row pointers were scanned; then s_ptr_copy (nblk_r + 1 ints of LDS) holds them.
constexpr int SDD_BALANCE_MAX_ROWS = 1024;
static __device__ __forceinline__ bool sdd_band_rows(const int32_t* __restrict__ ptr, int nnz, int nblk_r, int tiles_r, int band,
                                                     int SR, bool even, int band_room, int* s_rowid, int* scratch, int tid, int nthreads,
                                                     int* s_ptr_copy) {
    bool skewed = false;
    const int pairs = (nblk_r + 1) / 2;
    const float per_band = __builtin_amdgcn_rcpf((float)tiles_r);
    // (even bands in whole pairs of rows: 128 bytes of G.  Up to 512 pairs and as many bands the quotient is that of the integers)
    auto first_row = [&](int b) {
        return !even ? b * SR : 2 * (nblk_r <= SDD_BALANCE_MAX_ROWS ? (int)(((float)(pairs * b) + 0.5f) * per_band) : (int)((long long)pairs * b / tiles_r));
    };
    const bool scanned = nblk_r <= SDD_BALANCE_MAX_ROWS && tiles_r >= 2;
    if (scanned) {
        for (int r = tid; r < nblk_r; r += nthreads) {
            const int lo = clamp_entry(ptr[r], nnz), hi = clamp_entry(ptr[r + 1], nnz);
            s_ptr_copy[r] = lo;   // saves the caller a second trip to global memory
            if (r == nblk_r - 1) s_ptr_copy[nblk_r] = hi;
            scratch[r] = hi > lo ? hi - lo : 0;
        }
        __syncthreads();
        // (every wave for itself: as atomics on two words the lanes of a wave take turns, 10500 cycles for 128 rows instead of 2300)
        int most = 0, sum = 0, fullest = 0;
        if (even)
            for (int b = tid & 63; b < tiles_r; b += 64) {
                const int hi = first_row(b + 1);
                const int n = s_ptr_copy[hi < nblk_r ? hi : nblk_r] - s_ptr_copy[first_row(b)];
                fullest = n > fullest ? n : fullest;
            }
        for (int r = tid & 63; r < nblk_r; r += 64) {
            const int n = scratch[r];
            most = n > most ? n : most;
            sum += n;
        }
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) {
            const int m = __shfl_xor(most, d), f = __shfl_xor(fullest, d);
            most = m > most ? m : most;
            fullest = f > fullest ? f : fullest;
            sum += __shfl_xor(sum, d);
        }
        skewed = (long long)most * nblk_r > 2ll * sum || (even && fullest > band_room);
    }
    if (tid < SR) {
        const int lo = first_row(band), hi = even ? first_row(band + 1) : lo + SR, r = lo + tid;
        s_rowid[tid] = (!skewed && r < hi && r < nblk_r) ? r : -1;
    }
    __syncthreads();
    if (skewed) {
        for (int r = tid; r < nblk_r; r += nthreads) {
            const int n = scratch[r];
            int rank = 0;
            for (int o = 0; o < nblk_r; ++o) {
                const int m = scratch[o];
                rank += (m > n || (m == n && o < r)) ? 1 : 0;
            }
            const int place = rank / tiles_r;
            int b = rank % tiles_r;
            if (place & 1) b = tiles_r - 1 - b;
            if (b == band && place < SR) s_rowid[place] = r;
        }
        __syncthreads();
    }
    return scanned;
}

// Sums of the token slices, in slice order: n values of the blocks and, behind them, total - n of the bias (both multiples
// of 4).  Bound by the bytes of the partial sums; eight loads of a thread in flight
// (one at a time: 16 slices of 256 blocks 9.9 us instead of 7.3).
template <typename T>
static __device__ __forceinline__ void sdd_reduce(const float* partial, T* out, size_t n, T* bias_out, size_t total, int nsplit, unsigned block) {
    using E = Elem<T>;
    const size_t i4 = ((size_t)block * 256 + threadIdx.x) * 4;
    if (i4 >= total) return;
    // non-temporal loads: the partial sums are not read again
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    f32x4 s = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(partial + i4));
#pragma unroll 8
    for (int k = 1; k < nsplit; ++k) s += __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(partial + (size_t)k * total + i4));
    T* o = i4 < n ? out + i4 : bias_out + (i4 - n);
    o[0] = E::from_f32(s.x);
    o[1] = E::from_f32(s.y);
    o[2] = E::from_f32(s.z);
    o[3] = E::from_f32(s.w);
}
template <typename T>
__global__ __launch_bounds__(256) void sdd_reduce_kernel(const float* partial, T* out, size_t n, T* bias_out, size_t total, int nsplit) {
    sdd_reduce(partial, out, n, bias_out, total, nsplit, blockIdx.x);
}

}  // namespace pbs
