// Device-side build of the five int32 index arrays of a block mask.
//
// One workgroup of 1024 threads does the whole job (the grids are at most a few hundred thousand
// positions and this runs only when a pattern is created or changed).  Pass 1 walks the mask in
// row-major order: an exclusive scan of per-thread counts gives every nonzero its rank i, hence
// cols_a[i] = (col, block_ptr[i]), the row starts and blocks[block_ptr[i]] = (col, row).  Pass 2
// walks it in column-major order for rows_b / col_start_ends_b and finds each nonzero's data
// block by a binary search of its column in the (sorted) CSR row written by pass 1.
#pragma once
#include "pbs_common.h"

namespace pbs {

constexpr int INDEX_THREADS = 1024;

// exclusive scan of one int per thread over the workgroup; *total gets the sum
static __device__ int block_exclusive_scan(int v, int* s_wave /*[17]*/, int* total) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(incl, d, 64);
        if (lane >= d) incl += o;
    }
    __syncthreads();   // s_wave may still be read from a previous scan
    if (lane == 63) s_wave[wave] = incl;
    __syncthreads();
    if (tid == 0) {
        int run = 0;
        for (int w = 0; w < INDEX_THREADS / 64; ++w) {
            const int c = s_wave[w];
            s_wave[w] = run;
            run += c;
        }
        s_wave[16] = run;
    }
    __syncthreads();
    *total = s_wave[16];
    return s_wave[wave] + incl - v;
}

__global__ __launch_bounds__(INDEX_THREADS) void build_indices_kernel(
    const uint8_t* __restrict__ mask, const int64_t* __restrict__ block_ptr, int X, int Y, int nnz,
    int32_t* cols_a, int32_t* row_ptr, int32_t* rows_b, int32_t* col_ptr, int32_t* blocks, int32_t* status) {
    __shared__ int s_wave[17];
    __shared__ int s_err;
    const int tid = threadIdx.x;
    const long long total = (long long)X * Y;
    const long long chunk = (total + INDEX_THREADS - 1) / INDEX_THREADS;
    long long lo = tid * chunk, hi = lo + chunk;
    if (lo > total) lo = total;
    if (hi > total) hi = total;
    if (tid == 0) s_err = 0;

    // ---- pass 1: row-major ----
    int cnt = 0;
    for (long long p = lo; p < hi; ++p) cnt += mask[p] ? 1 : 0;
    int counted;
    int rank = block_exclusive_scan(cnt, s_wave, &counted);
    if (counted != nnz) {
        if (tid == 0) {
            status[0] = counted;
            status[1] = 1;
        }
        return;
    }
    for (long long p = lo; p < hi; ++p) {
        const int r = (int)(p / Y), c = (int)(p % Y);
        if (c == 0) row_ptr[r] = rank;
        if (mask[p]) {
            long long bp = block_ptr ? block_ptr[rank] : rank;
            if (bp < 0 || bp >= nnz) {
                s_err = 2;
                bp = -1;
            }
            cols_a[2 * rank] = c;
            cols_a[2 * rank + 1] = (int)bp;
            if (bp >= 0) {
                blocks[2 * bp] = c;
                blocks[2 * bp + 1] = r;
            }
            ++rank;
        }
    }
    if (tid == 0) row_ptr[X] = nnz;
    __threadfence();
    __syncthreads();

    // ---- pass 2: column-major ----
    cnt = 0;
    for (long long q = lo; q < hi; ++q) {
        const int c = (int)(q / X), r = (int)(q % X);
        cnt += mask[(long long)r * Y + c] ? 1 : 0;
    }
    rank = block_exclusive_scan(cnt, s_wave, &counted);
    for (long long q = lo; q < hi; ++q) {
        const int c = (int)(q / X), r = (int)(q % X);
        if (r == 0) col_ptr[c] = rank;
        if (mask[(long long)r * Y + c]) {
            int l = row_ptr[r], u = row_ptr[r + 1];
            while (l < u) {
                const int mid = (l + u) >> 1;
                if (cols_a[2 * mid] < c) l = mid + 1; else u = mid;
            }
            rows_b[2 * rank] = r;
            rows_b[2 * rank + 1] = cols_a[2 * l + 1];
            ++rank;
        }
    }
    if (tid == 0) col_ptr[Y] = nnz;
    __syncthreads();
    if (tid == 0) {
        status[0] = nnz;
        status[1] = s_err;
    }
}

// ---- the CSR pair of a pattern given as the reference's `blocks` list ----
// blocks[2 b] = block column, blocks[2 b + 1] = block row of data block b, in any order.  owner[p] = data block
// at row-major position p of the X x Y grid, or -1; then one row-major sweep of owner writes cols_a (sorted by
// row, then column) and the row starts.  A position listed twice keeps one of its data blocks (the other gets no
// result); entries outside the grid are skipped.
__global__ __launch_bounds__(256) void blocks_owner_clear_kernel(int* owner, long long total) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < total) owner[i] = -1;
}
__global__ __launch_bounds__(256) void blocks_owner_kernel(const int32_t* __restrict__ blocks, int nnz, int X, int Y, int* owner) {
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b >= nnz) return;
    const int c = blocks[2 * b], r = blocks[2 * b + 1];
    if (c >= 0 && c < Y && r >= 0 && r < X) owner[(long long)r * Y + c] = b;
}
__global__ __launch_bounds__(INDEX_THREADS) void csr_from_owner_kernel(const int* __restrict__ owner, int X, int Y,
                                                                       int32_t* cols_a, int32_t* row_ptr) {
    __shared__ int s_wave[17];
    const int tid = threadIdx.x;
    const long long total = (long long)X * Y;
    const long long chunk = (total + INDEX_THREADS - 1) / INDEX_THREADS;
    long long lo = tid * chunk, hi = lo + chunk;
    if (lo > total) lo = total;
    if (hi > total) hi = total;
    int cnt = 0;
    for (long long p = lo; p < hi; ++p) cnt += owner[p] >= 0 ? 1 : 0;
    int counted;
    int rank = block_exclusive_scan(cnt, s_wave, &counted);
    for (long long p = lo; p < hi; ++p) {
        const int r = (int)(p / Y), c = (int)(p % Y);
        if (c == 0) row_ptr[r] = rank;
        const int b = owner[p];
        if (b >= 0) {
            cols_a[2 * rank] = c;
            cols_a[2 * rank + 1] = b;
            ++rank;
        }
    }
    if (tid == 0) row_ptr[X] = counted;
}

// ---- move data blocks (block_replace): all five arrays from the old `blocks` list and a list of moves ----
// One workgroup, five short phases over the data blocks instead of scans over the grid: every block sets its bit in a bitmap
// of its row and in one of its column; a row's (column's) start is the sum of the popcounts before it, and a block's place within it
// the popcount of the bits below its own.  No sort, no search; the bitmaps sit in LDS while they fit (16 K positions take
// 4 KB, 24 x 96 positions and 1152 blocks 7 us in all, where building a mask, sorting the positions and the two scans of
// build_indices_kernel took 150 us in a dozen launches).
constexpr int REPLACE_LDS_WORDS = 12 * 1024;
enum ReplaceError { REPLACE_BAD_ID = 1, REPLACE_BAD_POSITION = 2, REPLACE_TAKEN = 4 };
static inline size_t replace_bitmap_words(int X, int Y) { return (size_t)X * ((Y + 31) / 32) + (size_t)Y * ((X + 31) / 32); }
static inline size_t replace_ws_bytes(int X, int Y, int nnz) {
    const size_t words = replace_bitmap_words(X, Y);
    return ((size_t)nnz + (words > REPLACE_LDS_WORDS ? words : 0)) * sizeof(int);
}
__global__ __launch_bounds__(INDEX_THREADS) void replace_blocks_kernel(
    const int32_t* __restrict__ old_blocks, const int64_t* __restrict__ moves, int n_moves, int X, int Y, int nnz, int32_t* cols_a,
    int32_t* row_ptr, int32_t* rows_b, int32_t* col_ptr, int32_t* blocks, int32_t* status, int* ws) {
    __shared__ unsigned s_bits[REPLACE_LDS_WORDS];
    __shared__ int s_wave[17];
    __shared__ int s_err;
    const int tid = threadIdx.x;
    const int wr = (Y + 31) / 32, wc = (X + 31) / 32;   // words per row, per column
    const int words = X * wr + Y * wc;
    int* pos = ws;                                      // [nnz] row-major position of every data block
    unsigned* bits = words > REPLACE_LDS_WORDS ? reinterpret_cast<unsigned*>(ws + nnz) : s_bits;
    unsigned* row_bits = bits;
    unsigned* col_bits = bits + (size_t)X * wr;
    if (tid == 0) s_err = 0;
    for (int i = tid; i < words; i += INDEX_THREADS) bits[i] = 0u;
    for (int b = tid; b < nnz; b += INDEX_THREADS) {
        const int c = old_blocks[2 * b], r = old_blocks[2 * b + 1];
        pos[b] = c >= 0 && c < Y && r >= 0 && r < X ? r * Y + c : -1;
    }
    __threadfence_block();
    __syncthreads();
    for (int i = tid; i < n_moves; i += INDEX_THREADS) {
        const int64_t r = moves[3 * (size_t)i], c = moves[3 * (size_t)i + 1], b = moves[3 * (size_t)i + 2];
        if (b < 0 || b >= nnz) atomicOr(&s_err, REPLACE_BAD_ID);
        else pos[b] = r >= 0 && r < X && c >= 0 && c < Y ? (int)(r * Y + c) : -1;
    }
    __threadfence_block();
    __syncthreads();
    for (int b = tid; b < nnz; b += INDEX_THREADS) {
        const int p = pos[b];
        if (p < 0) {
            atomicOr(&s_err, REPLACE_BAD_POSITION);
            continue;
        }
        const int r = p / Y, c = p - r * Y;
        const unsigned was = atomicOr(&row_bits[(size_t)r * wr + (c >> 5)], 1u << (c & 31));
        if ((was >> (c & 31)) & 1u) atomicOr(&s_err, REPLACE_TAKEN);
        atomicOr(&col_bits[(size_t)c * wc + (r >> 5)], 1u << (r & 31));
    }
    __threadfence_block();
    __syncthreads();
    // (the host may be waiting for the word and not for the kernel: it comes behind all that it stands for.  Every wave waits until its stores are in the L2 of
    // their common XCD, one thread writes that back for the others; a fence of all threads takes the kernel from 7 to 12 us)
    auto report = [&](int value) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0) {
            __threadfence();
            __hip_atomic_store(status, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    };
    if (s_err) {   // the same for every thread
        report(s_err);
        return;
    }
    auto starts = [&](const unsigned* line, int n, int w, int32_t* ptr) {
        int carry = 0;
        for (int base = 0; base < n; base += INDEX_THREADS) {
            const int i = base + tid;
            int cnt = 0;
            if (i < n)
                for (int k = 0; k < w; ++k) cnt += __popc(line[(size_t)i * w + k]);
            int total;
            const int before = block_exclusive_scan(cnt, s_wave, &total);
            if (i < n) ptr[i] = carry + before;
            carry += total;
        }
        if (tid == 0) ptr[n] = carry;
    };
    starts(row_bits, X, wr, row_ptr);
    starts(col_bits, Y, wc, col_ptr);
    __threadfence_block();
    __syncthreads();
    auto below = [](const unsigned* line, int at) {
        int n = __popc(line[at >> 5] & ((1u << (at & 31)) - 1u));
        for (int k = 0; k < at >> 5; ++k) n += __popc(line[k]);
        return n;
    };
    for (int b = tid; b < nnz; b += INDEX_THREADS) {
        const int p = pos[b], r = p / Y, c = p - r * Y;
        const int i = row_ptr[r] + below(row_bits + (size_t)r * wr, c), j = col_ptr[c] + below(col_bits + (size_t)c * wc, r);
        reinterpret_cast<int2*>(cols_a)[i] = make_int2(c, b);
        reinterpret_cast<int2*>(rows_b)[j] = make_int2(r, b);
        reinterpret_cast<int2*>(blocks)[b] = make_int2(c, r);
    }
    report(0);
}

// ---- consistency of the five arrays, one bit of *status per broken condition (PBS_BAD_* in pbs_hip.h) ----
// One workgroup; every index is checked before it is used, so any contents are safe to look at.  (The same checks as some
// seventy tensor operations took 0.5 ms of launches.)
static inline size_t validate_ws_bytes(int nnz) { return (size_t)nnz * 6 * sizeof(int); }
__global__ __launch_bounds__(INDEX_THREADS) void validate_indices_kernel(
    const int32_t* __restrict__ cols_a, const int32_t* __restrict__ row_ptr, const int32_t* __restrict__ rows_b,
    const int32_t* __restrict__ col_ptr, const int32_t* __restrict__ blocks, int X, int Y, int nnz, int32_t* status, int* ws) {
    __shared__ int s_bad;
    const int tid = threadIdx.x;
    int* seen[2] = {ws, ws + nnz};                                   // times a data block is listed
    int2* at[2] = {reinterpret_cast<int2*>(ws + 2 * (size_t)nnz), reinterpret_cast<int2*>(ws + 4 * (size_t)nnz)};   // (list, coordinate) of it
    if (tid == 0) s_bad = 0;
    for (int b = tid; b < nnz; b += INDEX_THREADS) {
        seen[0][b] = seen[1][b] = 0;
        at[0][b] = at[1][b] = make_int2(-1, -1);
    }
    __threadfence_block();
    __syncthreads();
    int bad = 0;
    auto list = [&](int which, const int32_t* ids, const int32_t* ends, int lists, int limit) {
        const int base = 4 * which;
        for (int i = tid; i <= lists; i += INDEX_THREADS) {
            const int e = ends[i];
            if (i == 0 ? e != 0 : e < ends[i - 1]) bad |= PBS_BAD_ROW_STARTS << base;
            if (i == lists && e != nnz) bad |= PBS_BAD_ROW_END << base;
        }
        auto owner = [&](int e) {   // the list that entry e belongs to: the last one that starts at or before it
            int lo = 0, hi = lists;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (ends[mid + 1] <= e) lo = mid + 1; else hi = mid;
            }
            return lo;
        };
        for (int e = tid; e < nnz; e += INDEX_THREADS) {
            const int c = ids[2 * (size_t)e], b = ids[2 * (size_t)e + 1], o = owner(e);
            if (c < 0 || c >= limit) bad |= PBS_BAD_COLS << base;
            if (e > 0 && o == owner(e - 1) && c <= ids[2 * (size_t)e - 2]) bad |= which ? PBS_BAD_ROWS_ORDER : PBS_BAD_COLS_ORDER;
            if (b < 0 || b >= nnz) {
                bad |= PBS_BAD_COLS_IDS << base;
            } else {
                atomicAdd(&seen[which][b], 1);
                at[which][b] = make_int2(o, c);
            }
        }
    };
    list(0, cols_a, row_ptr, X, Y);
    list(1, rows_b, col_ptr, Y, X);
    __threadfence_block();
    __syncthreads();
    for (int b = tid; b < nnz; b += INDEX_THREADS) {
        if (seen[0][b] != 1) bad |= PBS_BAD_COLS_IDS;
        if (seen[1][b] != 1) bad |= PBS_BAD_COLS_IDS << 4;
        const int2 a = at[0][b], t = at[1][b];   // (row, column), (column, row)
        if (a.x != t.y || a.y != t.x) bad |= PBS_BAD_LISTS_DIFFER;
        const int c = blocks[2 * (size_t)b], r = blocks[2 * (size_t)b + 1];
        if (c < 0 || c >= Y || r < 0 || r >= X) bad |= PBS_BAD_BLOCKS;
        if (c != a.y || r != a.x) bad |= PBS_BAD_BLOCKS_DIFFER;
    }
    if (bad) atomicOr(&s_bad, bad);
    __syncthreads();
    if (tid == 0) __hip_atomic_store(status, s_bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// out[c][r] = in[r][c] for a rows x cols matrix of 2- or 4-byte elements (tiles of 32 x 32 through LDS)
template <typename U>
__global__ __launch_bounds__(256) void transpose_dense_kernel(const U* __restrict__ in, U* __restrict__ out, long long rows,
                                                              long long cols) {
    __shared__ U s[32][33];
    const long long r0 = (long long)blockIdx.y * 32, c0 = (long long)blockIdx.x * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // 32 x 8
#pragma unroll
    for (int i = 0; i < 32; i += 8) {
        const long long r = r0 + ty + i, c = c0 + tx;
        if (r < rows && c < cols) s[ty + i][tx] = in[r * cols + c];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 32; i += 8) {
        const long long c = c0 + ty + i, r = r0 + tx;
        if (r < rows && c < cols) out[c * rows + r] = s[tx][ty + i];
    }
}

}  // namespace pbs
