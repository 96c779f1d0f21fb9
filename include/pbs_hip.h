/*
 * pbs_hip.h -- C ABI of libpbs_hip.so, the MI355X (gfx950) block-sparse matmul engine.
 *
 * Plain C: raw device pointers, sizes and a hipStream_t passed as void*.  No torch
 * types.  All pointers are caller-owned device memory; the library keeps nothing
 * after a call returns, so calls on different streams or from different host threads
 * do not interfere.  Its only device state of its own: the scratch array of the entry
 * point that allocates nothing (see there) and one diagnostic counter.
 *
 * Every entry point returns an int: 0 on success, a positive hipError_t when the HIP
 * runtime reported an error, a negative PBS_ERR_* when an argument was rejected
 * before anything was launched.  pbs_error_string() turns either into text.
 *
 * Data conventions (those of the reference's BlockSparseMatrix, block_sparse.py):
 *   - the weight W is [out_features, in_features], tiled in 32x32 blocks; X = out/32
 *     block rows, Y = in/32 block columns, nnz nonzero blocks;
 *   - packed data is [nnz*32, 32] row-major; data block b holds its W block
 *     transposed: data[32b + j][i] = W[32r + i][32c + j]      (block_sparse.py:326-331)
 *   - row_start_ends_a [X+1], cols_a [nnz][2] = (block col, data block)   CSR
 *   - col_start_ends_b [Y+1], rows_b [nnz][2] = (block row, data block)   CSC
 *   - blocks [nnz][2] = (block col, block row) of data block b         (:138-141)
 *   - dense operands are row-major and contiguous; dense results are row-major.
 */
#ifndef PBS_HIP_H
#define PBS_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define PBS_ABI_VERSION 10
#define PBS_BLOCK 32

/* element type of dense operands, packed data and results (accumulation is fp32) */
#define PBS_DTYPE_F32 0
#define PBS_DTYPE_BF16 1

#define PBS_OK 0
#define PBS_ERR_NULL_POINTER (-1)
#define PBS_ERR_BAD_SHAPE (-2)     /* negative size or a feature dim not a multiple of 32 */
#define PBS_ERR_BAD_DTYPE (-3)
#define PBS_ERR_MISALIGNED (-4)    /* a dense/data pointer is not 16-byte aligned */
#define PBS_ERR_WORKSPACE (-5)     /* workspace/plan buffer missing, misaligned or too small */
#define PBS_ERR_TOO_LARGE (-6)     /* a size exceeds what the kernels index with */
#define PBS_ERR_SCRATCH (-7)       /* more scratch needed than the built-in buffer of the no-allocation entry point */

int pbs_abi_version(void);
const char* pbs_error_string(int code);

/*
 * Index arrays of a block mask, built on the device, bit-exact with the reference's
 * BlockSparseMatrixBase.build_indices (block_sparse.py:125-153, helper :85-123).
 *
 *   mask       [X*Y] bytes, row-major, nonzero = block present
 *   block_ptr  NULL, or [nnz] int64: data-block id of the i-th nonzero in row-major
 *              order (the "recycled blocks" path used by block_replace, :210-219)
 *   nnz        the number of blocks the caller allocated outputs for
 *   status     [2] int32 device words: status[0] = number of nonzeros counted in mask,
 *              status[1] = 0 if ok, 1 if the count differs from nnz (nothing else is
 *              written then), 2 if a block_ptr entry is outside [0, nnz)
 */
int pbs_build_indices(const uint8_t* mask, const int64_t* block_ptr, int X, int Y, int nnz,
                      int32_t* cols_a, int32_t* row_start_ends_a,
                      int32_t* rows_b, int32_t* col_start_ends_b,
                      int32_t* blocks, int32_t* status, void* stream);

/*
 * Move data blocks to other positions and write all five index arrays again, in one launch
 * (BlockSparseMatrixBase.block_replace, block_sparse.py:167-219).
 *
 *   old_blocks [2*nnz]  the present `blocks` array
 *   moves   [n_moves,3] int64: (block row, block column, data block)
 *   status     one int32 word the GPU can write (device or pinned host memory): 0, or a sum of 1 (a data block outside
 *              [0, nnz)), 2 (a position outside the grid), 4 (two blocks at one position); nothing else is written then
 *   workspace  pbs_replace_blocks_workspace_bytes(X, Y, nnz) bytes of device memory
 */
size_t pbs_replace_blocks_workspace_bytes(int X, int Y, int nnz);
int pbs_replace_blocks(const int32_t* old_blocks, const int64_t* moves, int n_moves, int X, int Y, int nnz,
                       int32_t* cols_a, int32_t* row_start_ends_a, int32_t* rows_b, int32_t* col_start_ends_b,
                       int32_t* blocks, int32_t* status, void* workspace, size_t workspace_bytes, void* stream);

/*
 * Consistency of the five index arrays (sanity_check, block_sparse.py:431-463, and what the kernels rely on beyond it).
 * `status` as above: a sum of the bits below; the conditions of rows_b / col_start_ends_b have those of cols_a /
 * row_start_ends_a times 16.
 */
#define PBS_BAD_ROW_STARTS 1       /* does not start at 0, or decreases */
#define PBS_BAD_ROW_END 2          /* the last one is not nnz */
#define PBS_BAD_COLS 4             /* a coordinate outside the grid */
#define PBS_BAD_COLS_IDS 8         /* the data blocks are not a permutation */
#define PBS_BAD_BLOCKS 256         /* a position of `blocks` outside the grid */
#define PBS_BAD_COLS_ORDER 512     /* the coordinates of a list do not increase: cols_a */
#define PBS_BAD_ROWS_ORDER 1024    /* ... rows_b */
#define PBS_BAD_LISTS_DIFFER 2048  /* cols_a and rows_b hold different blocks */
#define PBS_BAD_BLOCKS_DIFFER 4096 /* `blocks` and cols_a hold different blocks */
size_t pbs_validate_indices_workspace_bytes(int nnz);
int pbs_validate_indices(const int32_t* cols_a, const int32_t* row_start_ends_a, const int32_t* rows_b,
                         const int32_t* col_start_ends_b, const int32_t* blocks, int X, int Y, int nnz,
                         int32_t* status, void* workspace, size_t workspace_bytes, void* stream);

/*
 * Schedule ("plan") of the dense x block-sparse product for one pattern and one direction.
 * It depends only on the index arrays, not on the data: build it when the pattern is created or
 * changed and pass it to every pbs_blocksparse_matmul call of that direction.  It is what the
 * reference's kernel derives again in every thread block from ptr/indices
 * (cutlass/gemm/block_loader_crosswise_prune_dense.h:254-264, :398-444), hoisted out of the hot
 * path: per result block column the list of its blocks, longest column first, and, for the bf16 kernels
 * with shared operand panels, the merged lists of groups of 16 columns.
 *
 *   transpose = 1 (forward):        ptr = row_start_ends_a, indices = cols_a, n = out, k = in
 *   transpose = 0 (input gradient): ptr = col_start_ends_b, indices = rows_b, n = in,  k = out
 *   (the coordinates increase within each list, as pbs_build_indices writes them; an entry whose coordinate or data
 *   block is outside its range is left out, and of several with one coordinate one is taken)
 *   plan: 16-byte aligned device buffer of pbs_blocksparse_matmul_plan_bytes(n, k) bytes
 */
size_t pbs_blocksparse_matmul_plan_bytes(int n, int k);
int pbs_blocksparse_matmul_plan(const int32_t* ptr, const int32_t* indices, int n, int k, int nnz,
                                void* plan, size_t plan_bytes, void* stream);

/*
 * The plan in parts, for callers whose pattern changes often: a product reads one part only, and the first
 * (PBS_PLAN_LIST, one launch) is all that fp32 and small bf16 products need.  `part` is a sum of PBS_PLAN_*;
 * pbs_blocksparse_matmul_part() tells which part a product of these sizes reads, given whether the call has a
 * workspace.  PBS_PLAN_LIST has to be there in any case.  pbs_blocksparse_matmul_plan builds everything.
 * Such a plan takes pbs_blocksparse_matmul_plan_part_bytes(n, k) bytes, about half of pbs_blocksparse_matmul_plan_bytes(n, k)
 * (a larger buffer will do as well).
 */
#define PBS_PLAN_LIST 1
#define PBS_PLAN_WIDE 2
#define PBS_PLAN_COLUMN 4
size_t pbs_blocksparse_matmul_plan_part_bytes(int n, int k);
int pbs_blocksparse_matmul_plan_part(const int32_t* ptr, const int32_t* indices, int n, int k, int nnz, int part,
                                     void* plan, size_t plan_bytes, void* stream);
int pbs_blocksparse_matmul_part(int64_t tokens, int n, int k, int nnz, int transpose, int dtype, int with_workspace);

/*
 * What a training step derives from a pattern, in one launch: the PBS_PLAN_LIST part of the plans of both directions (forward:
 * of the transposed weight) and, if `units` is not NULL, the unit table of the weight gradient
 * (pbs_blocksparse_matmul_back_units).  Same results and buffers as the calls that make them one by one; the plans take
 * pbs_blocksparse_matmul_plan_part_bytes.
 */
int pbs_blocksparse_derive(const int32_t* row_start_ends_a, const int32_t* cols_a, const int32_t* col_start_ends_b,
                           const int32_t* rows_b, int out_features, int in_features, int nnz, void* plan_forward,
                           size_t plan_forward_bytes, void* plan_input, size_t plan_input_bytes, void* units,
                           size_t units_bytes, void* stream);

/*
 * dense x block-sparse -> dense.  Replaces blocksparse_matmul_cutlass
 * (native/block_sparse_native.cpp:6-16, launcher native/block_sparse_cutlass_kernel.cu:113-150)
 * as called by BlockSparseMatrixBase.reverse_matmul_ (block_sparse.py:496-578).
 *
 *   transpose = 1 : out[tokens, n] = a[tokens, k] . W^T   n = out_features, k = in_features  (:518-521)
 *   transpose = 0 : out[tokens, n] = a[tokens, k] . W     n = in_features,  k = out_features (:522-525)
 *   plan: built by pbs_blocksparse_matmul_plan from the (ptr, indices) pair the reference passes
 *         here, for the same transpose
 *
 * Differences from the reference entry point, all on purpose: `data` is always the packed data as
 * stored (no per-call transposed copy of the weights, :541-544); `out` is row-major [tokens, n]
 * and need not be zeroed (the reference wants a zeroed [n, tokens] buffer, :516); `bias` is NULL
 * or [n] and is added in the epilogue (the reference adds it in a separate pass,
 * block_sparse_linear.py:231-232); any tokens >= 0 is handled; work is launched on `stream`,
 * not on stream 0.
 */
int pbs_blocksparse_matmul(const void* dense_a, const void* data, const void* plan,
                           const void* bias, void* dense_out,
                           int64_t tokens, int n, int k, int nnz,
                           int transpose, int dtype, void* stream);

/*
 * The same product with an optional workspace.  The reference's reverse_matmul_ hands its kernel a
 * transposed copy of the packed data for one of the two directions, made on every call
 * (block_sparse.py:541-544: data.reshape(-1, 32, 32).transpose(1, 2).reshape(-1, 32).contiguous()).
 * The fastest bf16 kernel for patterns with many blocks per column wants the same for the forward
 * direction (every block with the contraction index along its rows); the library makes that copy in
 * `workspace`, on `stream`, before the product, when the caller provides one of
 * pbs_blocksparse_matmul_workspace_bytes() bytes (16-byte aligned device memory, contents
 * unspecified afterwards).  With workspace = NULL, or one that is too small, the call is
 * pbs_blocksparse_matmul: same results to the last bit of bf16 rounding of the same fp32 sums in a
 * different order, from a kernel that reads the data as stored.  ..._workspace_bytes() returns 0 when
 * no copy would be made (fp32, the input-gradient direction, small or very sparse problems).
 *
 * Larger fp32 products run on the bf16 matrix cores, which multiply 16 times as fast: every value as the sum of three bfloat16 values
 * (without a rest), six of their nine products, sums in fp32.  The three products left out are at most 2^-24 of a product; a sum of many is closer to the
 * exact result than with fp32 instructions (1.1e-7 against 2.9e-7 of its size at 4096 x 4096, density 0.25), one of few nonzero products up to 1.4 times further off
 * (0.35e-7 against 0.25e-7).  For that the call writes the parts of the blocks into a workspace of pbs_blocksparse_matmul_parts_bytes() bytes (6 KB per block; 0
 * where such a workspace would not be used: bf16, smaller or very sparse problems).  Without it, the product is made of fp32 instructions.
 *
 * Bits.  A token's fp32 result is the same, to the last bit, in all calls of a pattern and direction that take the same of these two ways, whatever other
 * tokens share the call; between the two it differs by rounding.  Which way a call takes follows from its sizes: with the workspace the bf16 cores' from
 * 512 tokens and 2^21 tokens x blocks on at densities of 0.2 and more, apart from token counts for which an estimate sees the fp32 instructions ahead by a tenth
 * (pbs_blocksparse_matmul_parts_bytes() > 0 tells).  A caller who needs the same bits for requests batched in any way passes no workspace.  bf16
 * results, and the gradient of the blocks in either dtype, may differ by rounding between calls of different numbers of tokens.
 */
size_t pbs_blocksparse_matmul_workspace_bytes(int64_t tokens, int n, int k, int nnz, int transpose, int dtype);
size_t pbs_blocksparse_matmul_parts_bytes(int64_t tokens, int n, int k, int nnz, int transpose, int dtype);
int pbs_blocksparse_matmul_ws(const void* dense_a, const void* data, const void* plan,
                              const void* bias, void* dense_out,
                              int64_t tokens, int n, int k, int nnz,
                              int transpose, int dtype,
                              void* workspace, size_t workspace_bytes, void* stream);

/*
 * dense^T x dense -> block-sparse (only the nonzero blocks are computed), packed like
 * `data`:  out[32b + j][i] = sum_t dense_a[t][32r + i] * dense_b[t][32c + j].
 * Replaces blocksparse_matmul_back_cutlass (native/block_sparse_native.cpp:18-29,
 * launcher native/block_sparse_cutlass_kernel_back.cu:118-160) as called by
 * matmul_with_output_sparse_support_ (block_sparse.py:606-655); result layout as in
 * cutlass/gemm/block_task_back.h:537-538.
 *
 *   dense_a [tokens, out_features] (grad_output), dense_b [tokens, in_features] (input),
 *   both row-major contiguous.  The pattern is given by the CSR pair
 *   (row_start_ends_a, cols_a) instead of the reference's `blocks` list so that a
 *   workgroup can find the blocks of its tile of W without scanning all of them.
 *   A caller of the reference's entry point has the pair at hand: the object that owns
 *   `blocks` registers row_start_ends_a and cols_a as buffers next to it
 *   (block_sparse.py:58-65), built from the same mask by build_indices (:125-153); a
 *   caller that holds nothing but a mask obtains all of them from pbs_build_indices.
 *   Every token is accumulated (the reference drops tokens % 32 when tokens > 32).
 *   `out` need not be zeroed.
 *
 * When the blocks alone cannot fill the GPU the token range is split over workgroups and the fp32
 * partial blocks are summed in a fixed order by a second kernel; they and the unit table (below) lie
 * in `workspace`: pbs_blocksparse_matmul_back_workspace_bytes() bytes of 16-byte aligned device memory
 * (may be NULL when that returns 0).  In fp32 the partial blocks take at most 64 MiB, whatever the problem's size: ranges of
 * the tokens whose slices do not fit are added by further launches.
 *
 * Larger fp32 gradients run on the bf16 matrix cores, in three bfloat16 parts per value as above: where an estimate has that ahead, from 2^22 tokens x blocks on, and from
 * 2^20 on with 256 blocks and more (pbs_blocksparse_matmul_back_kernel_name() tells).  Between 2^20 and 2^22 the distance from the exact result is 0.69 times that of fp32 instructions on
 * average over 60 layers with normal operands (at most 0.83), 0.97 times where one input in ten is not zero (at most 1.18), and 1.12 times where a token has a single one (0.48e-7
 * of its size against 0.44e-7).
 */
size_t pbs_blocksparse_matmul_back_workspace_bytes(int64_t tokens, int out_features, int in_features,
                                                   int nnz, int dtype);
int pbs_blocksparse_matmul_back(const void* dense_a, const void* dense_b,
                                const int32_t* row_start_ends_a, const int32_t* cols_a,
                                void* data_out,
                                int64_t tokens, int out_features, int in_features, int nnz,
                                int dtype, void* workspace, size_t workspace_bytes, void* stream);

/*
 * The same product, and the bias gradient bias_out[n] = sum_t dense_a[t][n] (NULL: not wanted) from the same pass over
 * dense_a, for a caller that keeps what depends on the pattern alone.  No counterpart in the reference, which
 * sums the bias gradient on its own (block_sparse_linear.py:28-47).
 *
 *   units   the table of the work of the pattern's rows, made by pbs_blocksparse_matmul_back_units in
 *           pbs_blocksparse_matmul_back_units_bytes() bytes of 16-byte aligned device memory.  It depends on the
 *           pattern only and serves every number of tokens and both dtypes; some 160 bytes per block.  ..._units_bytes returns 0 for problems whose kernel uses
 *           none (units may then be NULL).
 *   workspace: pbs_blocksparse_matmul_back_bias_workspace_bytes() bytes, may be NULL when that is 0.
 *
 * nnz may be 0 with a bias_out; data_out may then be NULL.
 */
size_t pbs_blocksparse_matmul_back_units_bytes(int64_t tokens, int out_features, int in_features, int nnz, int dtype);
int pbs_blocksparse_matmul_back_units(const int32_t* row_start_ends_a, const int32_t* cols_a, int out_features, int in_features,
                                      int nnz, void* units, size_t units_bytes, void* stream);
size_t pbs_blocksparse_matmul_back_bias_workspace_bytes(int64_t tokens, int out_features, int in_features, int nnz,
                                                        int dtype);
int pbs_blocksparse_matmul_back_bias(const void* dense_a, const void* dense_b,
                                     const int32_t* row_start_ends_a, const int32_t* cols_a, const void* units,
                                     void* data_out, void* bias_out,
                                     int64_t tokens, int out_features, int in_features, int nnz,
                                     int dtype, void* workspace, size_t workspace_bytes, void* stream);

/*
 * The gradients of a linear layer's input, blocks and bias (bias_out may be NULL) in one call: pbs_blocksparse_matmul_ws with
 * transpose = 0 of grad_output and pbs_blocksparse_matmul_back_bias of grad_output and input, the same results bit for bit, with the
 * work in front of one product done by a launch of the other where both have any.
 *
 *   plan_input  the plan of (col_start_ends_b, rows_b), as for transpose = 0
 *   units, data_out, bias_out as above; grad_input [tokens, in_features]
 *   workspace   pbs_blocksparse_linear_back_workspace_bytes() bytes, 16-byte aligned, may be NULL when that is 0.  It holds what both products ask for at
 *               once: in fp32 up to 64 MiB of partial blocks and the blocks in parts, 6 KB each
 */
size_t pbs_blocksparse_linear_back_workspace_bytes(int64_t tokens, int out_features, int in_features, int nnz, int dtype);
int pbs_blocksparse_linear_back(const void* grad_output, const void* input, const void* data, const void* plan_input,
                                const int32_t* row_start_ends_a, const int32_t* cols_a, const void* units,
                                void* grad_input, void* data_out, void* bias_out,
                                int64_t tokens, int out_features, int in_features, int nnz,
                                int dtype, void* workspace, size_t workspace_bytes, void* stream);

/*
 * The same product with the arguments of the reference's entry point blocksparse_matmul_back_cutlass
 * (native/block_sparse_native.cpp:18-29; launcher native/block_sparse_cutlass_kernel_back.cu:118-160, which
 * picks one of four kernels by the two memory-order flags, :145-157), for a caller that holds what the
 * reference's call site holds (block_sparse.py:606-652): the two dense operands with a flag each, and the
 * `blocks` list.
 *
 *   a_row_major / b_row_major   1: the operand is [tokens, features] row-major (a "contiguous" torch tensor, the
 *                               reference's pytorch_contiguous_* = true); 0: it is [features, tokens] row-major,
 *                               i.e. its transpose is contiguous (block_sparse.py:480-494)
 *   blocks [nnz][2]             (block column, block row) of data block b, in any order (block_sparse.py:138-141)
 *
 * The CSR pair is derived from `blocks` on the device (three small kernels), and an operand given in the second
 * order is transposed on the device, both into `workspace`; then pbs_blocksparse_matmul_back runs.  All of it
 * is launched on `stream`.  workspace: 16-byte aligned device memory of
 * pbs_blocksparse_matmul_back_blocks_workspace_bytes() bytes (index arrays + transposed operands + the partial
 * sums of a split token range).  A caller that already holds row_start_ends_a / cols_a and row-major operands
 * saves those steps by calling pbs_blocksparse_matmul_back.
 */
size_t pbs_blocksparse_matmul_back_blocks_workspace_bytes(int64_t tokens, int out_features, int in_features, int nnz,
                                                          int dtype, int a_row_major, int b_row_major);
int pbs_blocksparse_matmul_back_blocks(const void* dense_a, int a_row_major, const void* dense_b, int b_row_major,
                                       void* data_out,
                                       int64_t tokens, int out_features, int in_features,
                                       const int32_t* blocks, int nnz,
                                       int dtype, void* workspace, size_t workspace_bytes, void* stream);

/*
 * pbs_blocksparse_matmul_back for callers that cannot allocate device memory: code under HIP graph
 * capture, tight serving loops, harnesses that forbid hipMalloc.  It has no counterpart in the
 * reference.  Same arguments and kernels as pbs_blocksparse_matmul_back, and where that one's workspace would fit the array bit-identical
 * results, without the workspace pair: the fp32 partial sums of a split token range go to a device array of
 * PBS_NOALLOC_SCRATCH_BYTES (64 MiB) that is part of the library (every GPU the library is used on
 * holds its own copy until the process ends).  The call makes no hipMalloc/hipFree and calls no
 * allocating routine.
 *
 *   - A problem of the row kernel whose pbs_blocksparse_matmul_back_workspace_bytes() exceeds the array runs with fewer slices
 *     of the tokens and more launches (the last bits of its sums may differ); one of the rectangle kernel is rejected with PBS_ERR_SCRATCH before anything is launched (4096 x 4096 at density 0.25 with 16384
 *     tokens in bf16 needs exactly 64 MiB and fits).
 *   - Nothing in the array has to be cleared between calls: every word the reduction kernel reads
 *     is written by the product kernel of the same call first.
 *   - All calls on one GPU share that GPU's array, whatever their stream: two calls that overlap on
 *     one GPU race.  Order them on one stream, or use the workspace entry point for concurrent work.
 *   - The first call on a GPU looks up that GPU's address of the array (hipGetSymbolAddress).  A caller that is
 *     going to capture the call into a HIP graph calls pbs_blocksparse_matmul_back_noalloc_init() once per GPU,
 *     with that GPU current, before the capture begins; it does the lookup and nothing else.
 */
#define PBS_NOALLOC_SCRATCH_BYTES (64u << 20)
size_t pbs_blocksparse_matmul_back_noalloc_max_bytes(void);
int pbs_blocksparse_matmul_back_noalloc_init(void);
int pbs_blocksparse_matmul_back_noalloc(const void* dense_a, const void* dense_b,
                                        const int32_t* row_start_ends_a, const int32_t* cols_a,
                                        void* data_out,
                                        int64_t tokens, int out_features, int in_features, int nnz,
                                        int dtype, void* stream);

/*
 * Diagnostics.  None has a counterpart in the reference.
 *
 * pbs_protocol_failures: the kernels for large problems (dds16_kernel, ddsc_kernel, split_kernel) synchronise their waves
 * through progress words in LDS with bounded waits instead of barriers.  A wait that runs into its bound means a
 * broken protocol; the kernel then writes NaN into the results it could not vouch for and counts the event in a
 * device word.  This call copies the current GPU's count (since the library was loaded) to *count; it synchronises
 * the device.  The Python layer checks it after every product when PBS_DEBUG is set and raises.
 *
 * pbs_blocksparse_matmul_kernel_name / ..._back_kernel_name: which kernel(s) a call with these sizes runs
 * ("stream_kernel", "walk_kernel", "split_kernel", "panel_kernel", "panel_chunk_kernel", "dds16_kernel", "ddsc_kernel"; "sdd_row_kernel", "sdd_split_kernel",
 * "sdd_bf16_kernel", with " + sdd_reduce_kernel" when the token range is split), for benchmark labels.  "" for arguments the product
 * entry points reject.
 *
 * pbs_blocksparse_matmul_kernel_form: that name and, behind a comma, what a test of a form of the kernel has to know: "lines ahead" where copies of
 * "ddsc_kernel" may ask for them.
 * pbs_blocksparse_matmul_back_kernel_form: of "sdd_bf16_kernel" its partition, as "11 even bands of 8 rows x 2 rectangles x 11 slices" ("even": of equal numbers of
 * rows, 8 at most).  The texts are the calling thread's until its next call.
 */
int pbs_protocol_failures(unsigned* count);
const char* pbs_blocksparse_matmul_kernel_name(int64_t tokens, int n, int k, int nnz, int transpose, int dtype,
                                               int with_workspace);
const char* pbs_blocksparse_matmul_kernel_form(int64_t tokens, int n, int k, int nnz, int transpose, int dtype,
                                               int with_workspace);
const char* pbs_blocksparse_matmul_back_kernel_name(int64_t tokens, int out_features, int in_features, int nnz,
                                                    int dtype);
const char* pbs_blocksparse_matmul_back_kernel_form(int64_t tokens, int out_features, int in_features, int nnz,
                                                    int dtype);

#ifdef __cplusplus
}
#endif
#endif /* PBS_HIP_H */
