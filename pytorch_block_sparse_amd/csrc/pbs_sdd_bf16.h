// bf16 weight gradient on the sparse support.
//
//   out[32b + j][i] = sum_t G[t][32r + i] * X[t][32c + j]   for every data block b at (r, c).
//
// One workgroup (8 waves) owns a rectangle of 16 x 16 or 8 x 16 block positions of W and one slice of the
// tokens.  The blocks present in the rectangle are listed row-major and dealt to the waves in equal
// contiguous runs (at most QW accumulators per wave; denser rectangles take further passes).
//
// Tokens are streamed in chunks of 32.  A chunk is 32 token rows of G (16 or 8 block rows, 1 KB or 512 bytes per
// token) and of X (16 block columns, 1 KB per token).  Both matrix operands need 8 consecutive tokens of a feature
// per lane, the rows hold consecutive features of a token.  So a lane loads the same eight features of eight token
// rows into registers, turns them there (a byte permutation per pair of values) and writes them to one of two chunk
// buffers as the operands themselves: a wave reads an operand with two ds_read_b128 of 1 KB each, at one address that an
// exclusive or makes from the block's place.  The loads are a chunk ahead of their writes, in two groups of four rows, so the texture path
// and the LDS's writes are busy in turn through the whole chunk.  Tokens past the slice's end are zeros by the loads' own
// bounds check.
//
// What it replaced copied the rows to the LDS as they are (one DMA instruction each) and read them with ds_read_b64_tr_b16, twice the LDS
// instructions at two thirds of their rate, in a loop of 60 instructions per block (12 now: no branch around a copied operand, no address
// arithmetic).  4096 -> 4096, 16384 tokens, with the reduction: density 0.25 216 -> 198 us, 0.5 (8 rows now) 428 -> 339; 768 -> 3072 density 0.5 112 -> 77;
// 2048 -> 2048 density 0.5 146 -> 105.  Of a chunk's 2500 cycles (16 rows, density 0.25) the matrix cores have 1024, the LDS 1300, the texture path
// 1450; the phases of the two waves of a SIMD overlap in part.  The chip is at its power limit (1.9 GHz): a build with 6 % fewer cycles took
// the same time.  Tried and not faster: the upper four waves two slots behind the lower four (210 us; 188 against 134 with few blocks: the waves no longer
// read a row of memory together), two barriers in the middle of a chunk instead of one at its start (212), eight rows of loads in one group
// (201), token-major rows through registers (228).
//
// The bias gradient (the sums of G's columns) comes out of the G panels in LDS: the rectangles of a band share the band's
// block rows among themselves.  4096 -> 4096 density 0.25, 16384 tokens: 3 us; a reduction of its own
// over G took 43 (the 134 MB of G once more).
//
// Consecutive blocks of a wave mostly share their block row, so the G operand is reloaded only when the row changes.
#pragma once
#include "pbs_common.h"
#include "pbs_sdd.h"

namespace pbs {

template <int SR_>
struct SddBf16Cfg {
    static constexpr int SR = SR_, SC = 16, NW = 8, NT = NW * 64, QW = 9;
    static constexpr int TC = 32;                            // tokens per chunk
    static constexpr int BLOCK_BYTES = TC * 64;              // a block row or column of a chunk
    static constexpr int X_PANEL = 32768, STAGE = 65536;     // offset of the X panel in a buffer, of the second buffer (powers of two: added by xor)
    static constexpr int LIST_MAX = SR * SC;
    static constexpr int QMAX = QW * NW;
    static constexpr int TABLE_BYTES = LIST_MAX * 4 + LIST_MAX * 2 + (2 * SR + SC / 2 + 4) * 4;
    static constexpr int LDS_BYTES = 2 * STAGE + TABLE_BYTES;
    static_assert(SR == 16 || SR == 8, "a G panel of 32 or 16 KB for four waves");
};

// The rectangle's rows, columns and block list, built by all threads of the workgroup (NT threads, of
// which the first 8 waves place the blocks).  smem: scratch of at least SDD_BF16_PROLOGUE_BYTES at the start
// of the (not yet used) chunk buffers.  Results in LDS: s_blk / s_pos (data block and (row place << 8 |
// column place) of each block, row-major), s_rowoff[SR] = number of blocks, s_rowid[SR] = block row of
// W in each row place or -1, s_gu[SC / 2] = column unit (pair of block columns) in each place or -1.
constexpr int SDD_BF16_EMAX = 8192, SDD_BF16_UMAX = 1024;
constexpr int SDD_BF16_PROLOGUE_BYTES = (2 * 16 + 1 + 2 * SDD_BF16_EMAX + 2 * SDD_BF16_UMAX + 2 * SDD_BALANCE_MAX_ROWS + 3) * 4;
template <int NT, int SR, typename Known>
static __device__ __forceinline__ void sdd_bf16_prologue(const SddArgs& a, int tile, unsigned char* smem, int* s_blk,
                                                         unsigned short* s_pos, int* s_rowoff, int* s_rowid, int* s_gu, Known&& known) {
    constexpr int SC = 16, NW = 8;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c0 = (tile % a.tiles_c) * SC;
    const int nblk_r = a.N / 32;
    // ---- which rows and columns of W this rectangle covers, and the list of its blocks (row-major) ----
    // Rows: the band's SR block rows (sdd_band_rows).  Columns: normally the band's columns c0 .. c0+15.
    // When the band's entries fit in LDS the columns of the band are instead dealt to the band's
    // rectangles by block count, in units of two adjacent columns (one 128-byte piece of an X row):
    // the units are ranked by their number of blocks in this band and handed out in serpentine order.
    // Rectangles of one band then hold the same number of blocks to within a few, instead of
    // 64 +- 7 at density 0.25, and the kernel no longer waits for its fullest rectangle.
    const int band = tile / a.tiles_c, grp = tile % a.tiles_c;
    const int nblk_c = a.K / 32;
    const int nunits = (nblk_c + 1) / 2;
    // scratch in the (not yet used) chunk buffers
    constexpr int EMAX = SDD_BF16_EMAX, UMAX = SDD_BF16_UMAX;
    int* s_lo = reinterpret_cast<int*>(smem);   // [SR] first entry of each row
    int* s_rs = s_lo + SR;                      // [SR + 1] start of each row's entries in the cached arrays
    int* s_ecol = s_rs + SR + 1;                // [EMAX] block column of each cached entry
    int* s_eblk = s_ecol + EMAX;                // [EMAX] data block of each cached entry
    int* s_cnt = s_eblk + EMAX;                 // [UMAX] blocks of the band per column unit
    int* s_ug = s_cnt + UMAX;                   // [UMAX] rectangle * 8 + place of each column unit
    int* s_scan = s_ug + UMAX;                  // [SDD_BALANCE_MAX_ROWS + 2] scratch of the row scan
    int* s_ptr_copy = s_scan + SDD_BALANCE_MAX_ROWS + 2;   // [SDD_BALANCE_MAX_ROWS + 1] row pointers, if scanned
    const bool have_ptr = sdd_band_rows(a.ptr, a.nnz, nblk_r, a.tiles_r, band, SR, a.even != 0, a.band_room, s_rowid, s_scan, tid, NT, s_ptr_copy);
    __syncthreads();
    if (tid < SR) {
        const int r = s_rowid[tid];
        int lo = 0, hi = 0;
        if (r >= 0) {
            if (have_ptr) {
                lo = s_ptr_copy[r];
                hi = s_ptr_copy[r + 1];
            } else {
                lo = clamp_entry(a.ptr[r], a.nnz);
                hi = clamp_entry(a.ptr[r + 1], a.nnz);
            }
        }
        s_lo[tid] = lo;
        s_rs[tid + 1] = hi > lo ? hi - lo : 0;
    }
    if (tid < SC / 2) s_gu[tid] = -1;
    __syncthreads();
    if (tid == 0) {
        int run = 0;
        s_rs[0] = 0;
        for (int i = 0; i < SR; ++i) {
            run += s_rs[i + 1];
            s_rs[i + 1] = run;
        }
    }
    __syncthreads();
    const int nent = s_rs[SR];
    const bool cached = nent <= EMAX;
    const bool dealt = cached && nunits <= UMAX && a.tiles_c >= 2;
    int my_lo = 0, my_n = 0;
    if (cached) {
        // one sweep over the band's entries (entry i belongs to the row r with s_rs[r] <= i < s_rs[r + 1]):
        // all loads of a thread are in flight together
        for (int i = tid; i < nent; i += NT) {
            int r = 0;
#pragma unroll
            for (int k = 1; k < SR; ++k) r += (i >= s_rs[k]) ? 1 : 0;
            const int2 e = *reinterpret_cast<const int2*>(a.idx + 2 * (size_t)(s_lo[r] + i - s_rs[r]));
            s_ecol[i] = e.x;
            s_eblk[i] = e.y;
        }
        if (dealt)
            for (int u = tid; u < nunits; u += NT) s_cnt[u] = s_ug[u] = 0;
        __syncthreads();
        if (dealt) {
            for (int i = tid; i < nent; i += NT) {
                const int c = s_ecol[i];
                if (c >= 0 && c < nblk_c) atomicAdd(&s_cnt[c >> 1], 1);
            }
            __syncthreads();
            // (the units that precede a unit, counted by several threads)
            const int parts = nunits < NT ? NT / nunits : 1, part = (nunits + parts - 1) / parts;
            for (int i = tid; i < parts * nunits; i += NT) {
                const int u = i % nunits, n = s_cnt[u], o0 = i / nunits * part, o1 = o0 + part < nunits ? o0 + part : nunits;
                int rank = 0;
#pragma unroll 4
                for (int o = o0; o < o1; ++o) {
                    const int m = s_cnt[o];
                    rank += (m > n || (m == n && o < u)) ? 1 : 0;
                }
                if (rank) atomicAdd(&s_ug[u], rank);
            }
            __syncthreads();
            for (int u = tid; u < nunits; u += NT) {
                const int rank = s_ug[u];
                const int place = rank / a.tiles_c;   // < SC / 2: there are at most 8 units per rectangle
                int gsel = rank % a.tiles_c;
                if (place & 1) gsel = a.tiles_c - 1 - gsel;
                s_ug[u] = gsel * (SC / 2) + place;
                if (gsel == grp) s_gu[place] = u;
            }
        } else if (tid < SC / 2) {
            const int u = grp * (SC / 2) + tid;
            s_gu[tid] = u < nunits ? u : -1;
        }
        __syncthreads();
        known();
        // rows 2*wave and 2*wave + 1: first count this rectangle's blocks, then (below) place them
        auto mine_of = [&](int c) -> int {   // place (0..15) of block column c in this rectangle, or -1
            if (c < 0 || c >= nblk_c) return -1;
            const int ug = dealt ? s_ug[c >> 1] : (c >> 1);
            return (ug / (SC / 2)) == grp ? (ug % (SC / 2)) * 2 + (c & 1) : -1;
        };
#pragma unroll
        for (int rr = 0; rr < SR / NW; ++rr) {
            if (wave >= NW) break;
            const int r = wave * (SR / NW) + rr;
            const int off = s_rs[r], n = s_rs[r + 1] - off;
            int cnt = 0;
            for (int b0 = 0; b0 < n; b0 += 64) {
                const bool m = (b0 + lane < n) && mine_of(s_ecol[off + b0 + lane]) >= 0;
                cnt += __popcll(__ballot(m));
            }
            if (lane == 0) s_rowoff[r] = cnt < SC ? cnt : SC;   // (repeated columns: never more than the tables hold)
        }
    } else {
        if (tid < SC / 2) {
            const int u = grp * (SC / 2) + tid;
            s_gu[tid] = u < nunits ? u : -1;
        }
        __syncthreads();
        known();
        if (tid < SR) {
            const int r = s_rowid[tid];
            if (r >= 0) {
                const int lo = clamp_entry(a.ptr[r], a.nnz), hi = clamp_entry(a.ptr[r + 1], a.nnz);
                int l = lo, u = hi;
                while (l < u) {   // rows are sorted by block column: first entry with column >= c0
                    const int mid = (l + u) >> 1;
                    if (a.idx[2 * mid] < c0) l = mid + 1; else u = mid;
                }
                my_lo = l;
                while (l < hi && a.idx[2 * l] < c0 + SC) ++l;
                my_n = l - my_lo;
                if (my_n > SC) my_n = SC;
            }
            s_rowoff[tid] = my_n;
        }
    }
    __syncthreads();
    if (tid == 0) {
        int run = 0;
        for (int i = 0; i < SR; ++i) {
            const int n = s_rowoff[i];
            s_rowoff[i] = run;
            run += n;
        }
        s_rowoff[SR] = run;
    }
    __syncthreads();
    if (cached) {
        auto mine_of = [&](int c) -> int {
            if (c < 0 || c >= nblk_c) return -1;
            const int ug = dealt ? s_ug[c >> 1] : (c >> 1);
            return (ug / (SC / 2)) == grp ? (ug % (SC / 2)) * 2 + (c & 1) : -1;
        };
#pragma unroll
        for (int rr = 0; rr < SR / NW; ++rr) {
            if (wave >= NW) break;
            const int r = wave * (SR / NW) + rr;
            const int off = s_rs[r], n = s_rs[r + 1] - off;
            int run = s_rowoff[r];
            for (int b0 = 0; b0 < n; b0 += 64) {
                const int cl = (b0 + lane < n) ? mine_of(s_ecol[off + b0 + lane]) : -1;
                const unsigned long long bal = __ballot(cl >= 0);
                const int at = run + __popcll(bal & ((1ull << lane) - 1ull));
                if (cl >= 0 && at < s_rowoff[r + 1]) {
                    int b = s_eblk[off + b0 + lane];
                    if (b < 0 || b >= a.nnz) b = -1;
                    s_blk[at] = b;
                    s_pos[at] = (unsigned short)((r << 8) | cl);
                }
                run += __popcll(bal);
            }
        }
    } else if (tid < SR) {
        const int off = s_rowoff[tid];
        for (int i = 0; i < my_n; ++i) {
            const int c = a.idx[2 * (my_lo + i)];
            int b = a.idx[2 * (my_lo + i) + 1];
            if (b < 0 || b >= a.nnz) b = -1;
            s_blk[off + i] = b;
            s_pos[off + i] = (unsigned short)((tid << 8) | (c - c0));
        }
    }
    __syncthreads();
}

// BIAS: with the bias gradient (bias_out given).  The build without it spares layers without a bias the bookkeeping of the sums (18
// spilled scalar registers instead of none).
template <bool BIAS, int SR>
static __device__ __forceinline__ void sdd_rectangle(const SddArgs& a) {
    using C = SddBf16Cfg<SR>;
    constexpr int NW = C::NW, TC = C::TC, QW = C::QW;

    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    int* s_blk = reinterpret_cast<int*>(smem + 2 * C::STAGE);                       // [LIST_MAX] data block
    unsigned short* s_pos = reinterpret_cast<unsigned short*>(s_blk + C::LIST_MAX);  // [LIST_MAX] (rl << 8) | cl
    int* s_rowoff = reinterpret_cast<int*>(s_pos + C::LIST_MAX);                     // [SR + 1]

    const int ntiles = a.tiles_r * a.tiles_c;
    const int wg = xcd_tile_id(blockIdx.x, ntiles * a.nsplit);
    if (wg < 0) return;
    const int sp = wg / ntiles;
    const int tile = wg % ntiles;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lrow = lane & 31;
    const int h = lane >> 5;

    // ---- which rows and columns of W this rectangle covers, and the list of its blocks (row-major) ----
    int* s_rowid = s_rowoff + SR + 2;   // [SR] block row of W in each place of this rectangle's band, or -1
    int* s_gu = s_rowid + SR;           // [SC / 2] column unit in each place of this rectangle, or -1
    static_assert(SDD_BF16_PROLOGUE_BYTES <= 2 * C::STAGE, "scratch fits in the chunk buffers");
    const int nblk_c = a.K / 32;
    const int t_begin = __builtin_amdgcn_readfirstlane(sp * a.tokens_per_split);
    const int t_end = t_begin + a.tokens_per_split < a.M ? t_begin + a.tokens_per_split : a.M;
    const int nchunks = t_begin < t_end ? (t_end - t_begin + TC - 1) / TC : 0;

    // ---- this wave's share of a chunk: the 16 bytes (eight features) at chunk position `pc` of eight token rows of G or of X in every
    //      lane, transposed in registers to eight tokens of each feature ----
    // Waves 0 to 3 copy X, a group of eight tokens each; the others G: with SR = 16 a group as well, with SR = 8 half of two groups.
    const bool of_g = wave >= NW / 2, whole = SR == 16 || !of_g;
    constexpr int G_LANES = SR * 4;
    const int pc = of_g ? lane % G_LANES : lane, place = pc >> 2;
    const int tg = SR == 16 || !of_g ? wave & 3 : (wave & 2) + lane / G_LANES;   // group of eight tokens
    const unsigned row_bytes = (unsigned)(of_g ? a.N : a.K) * 2;
    // Four rows at a time: in every other pair of places the last four of the eight first, so that the lanes that write together fill
    // whole 16-byte places of the LDS.
    const int half = ((place >> 1) ^ (whole ? 0 : wave)) & 1;
    unsigned voff = (unsigned)(8 * tg + 4 * half) * row_bytes;
    auto find_source = [&]() {
        // The 64 bytes of a place come from its block row of W, or block column (two adjacent columns per unit); a place without one
        // fetches any valid address; nothing reads it.
        int src;
        if (of_g) {
            src = s_rowid[place];
        } else {
            const int unit = s_gu[place >> 1];
            src = unit >= 0 ? unit * 2 + (place & 1) : -1;
            if (src >= nblk_c) src = -1;
        }
        if (src >= 0) voff += (unsigned)(src * 64 + (pc & 3) * 16);
    };
    // the chunk being loaded, as a buffer that ends with the slice: a load behind the end gives zeros and reads nothing
    const unsigned char* ld_base = nullptr;
    int ld_left = 0, ld_bytes = 0;   // tokens from the chunk being loaded to the end of the slice; bytes of its rows
    uint4 st[8];
    auto load_reset = [&]() {
        ld_base = static_cast<const unsigned char*>(of_g ? a.g : a.x) + (size_t)t_begin * row_bytes;
        ld_left = t_end - t_begin;
        ld_bytes = (ld_left < 0 ? 0 : (ld_left < TC ? ld_left : TC)) * row_bytes;
    };
    auto load_next = [&]() {
        ld_base = uniform_ptr(ld_base + (size_t)TC * row_bytes);   // (kept in scalar registers: each load is a loop otherwise)
        ld_left -= TC;
        ld_bytes = __builtin_amdgcn_readfirstlane((ld_left < 0 ? 0 : (ld_left < TC ? ld_left : TC)) * row_bytes);
    };
    const unsigned second = half ? 0u - 4 * row_bytes : 4 * row_bytes;
    auto load_row = [&](int k) {   // 0..3: the lane's first four rows, 4..7: the others
        unsigned step = (k & 3) * row_bytes;
        asm volatile("" : "+s"(step));   // (the offsets of all rows kept in vector registers spill)
        st[k] = buffer16(ld_base, k < 4 || whole ? ld_bytes : 0, voff + step + (k < 4 ? 0u : second));   // (no branch: the waits count loads)
    };
    // LDS: a block of a panel is its two matrix operands of 16 tokens, 1 KB each: 512 bytes for the first eight tokens, 512 for the
    // others, 16 per feature.  Bits 4..7 of an address are swizzled by bits of the lane that writes it: the lanes that write together
    // would otherwise meet in two places of 16 bytes, mod 256.
    const int write_at = (of_g ? 0 : C::X_PANEL) + place * C::BLOCK_BYTES + (tg >> 1) * 1024 + (tg & 1) * 512 +
                         (((pc & 3) * 128 + (pc & 3) * 16) ^ (place & 3) << 6) + half * 8;
    auto write_features = [&](int four, int d, int stage) {   // features 2d and 2d + 1 of the lane's first (0) or other (1) four rows
        const uint32_t r[4] = {(&st[4 * four].x)[d], (&st[4 * four + 1].x)[d], (&st[4 * four + 2].x)[d], (&st[4 * four + 3].x)[d]};
        const int at = write_at ^ stage ^ four << 3;
        *reinterpret_cast<uint2*>(smem + (at ^ (2 * d) << 4)) =
            make_uint2(__builtin_amdgcn_perm(r[1], r[0], 0x05040100u), __builtin_amdgcn_perm(r[3], r[2], 0x05040100u));
        *reinterpret_cast<uint2*>(smem + (at ^ (2 * d + 1) << 4)) =
            make_uint2(__builtin_amdgcn_perm(r[1], r[0], 0x07060302u), __builtin_amdgcn_perm(r[3], r[2], 0x07060302u));
    };

    // ---- fragment addresses: lane l serves feature l & 31 of the block; lane half h tokens 8h .. 8h + 7 of each 16-token matrix step ----
    const int read_at = h * 512 + (lrow & 24) * 16 + (((lrow & 7) ^ (lrow >> 3)) << 4);

    auto load_first = [&]() {
        load_reset();
#pragma unroll
        for (int k = 0; k < 8; ++k) load_row(k);
        load_next();
    };
    // (the first loads are on their way while the blocks are listed: with the row counts and ranks above 29000 -> 13500 cycles to the first product)
    sdd_bf16_prologue<C::NT, SR>(a, tile, smem, s_blk, s_pos, s_rowoff, s_rowid, s_gu, [&]() {
        find_source();
        load_first();
    });
    const int nq = __builtin_amdgcn_readfirstlane(s_rowoff[SR]);
    // bias gradient: places sum_p0 .. sum_p0 + sum_rows - 1 of the band are this rectangle's.  A thread sums one feature, over every
    // sum_step-th group of eight tokens.
    const int sum_share = (SR + a.tiles_c - 1) / a.tiles_c, sum_p0 = (tile % a.tiles_c) * sum_share;
    const int sum_rows = !BIAS || sum_p0 >= SR ? 0 : (sum_p0 + sum_share < SR ? sum_share : SR - sum_p0);
    if (nq == 0 && sum_rows == 0) return;
    const int sum_width = sum_rows > 0 ? 32 * sum_rows : 1, sum_step = C::NT / sum_width < 4 ? C::NT / sum_width : 4;
    const int sum_t0 = tid / sum_width, sum_place = sum_p0 + tid % sum_width / 32, sum_f = tid % 32;
    const bool sum_mine = sum_rows > 0 && sum_t0 < sum_step;
    float sum = 0.f;

    bf16_t* out = static_cast<bf16_t*>(a.out);
    float* part = a.partial ? a.partial + (size_t)sp * ((size_t)a.nnz * 1024 + (BIAS ? a.N : 0)) : nullptr;

    for (int q0 = 0; q0 < nq || (BIAS && q0 == 0); q0 += C::QMAX) {
        // this pass: blocks [q0, q0 + npass), dealt to the waves in contiguous runs
        const int npass = (nq - q0 < C::QMAX) ? nq - q0 : C::QMAX;
        // (runs of npass / NW blocks, the first npass % NW waves one more: with runs of ceil(npass / NW) the last
        // wave of 66 blocks had 3 and the others 9)
        const int per = npass / NW, rem = npass % NW;
        const int w_lo = q0 + wave * per + (wave < rem ? wave : rem);
        const int w_n = per + (wave < rem ? 1 : 0);

        // per accumulator slot: where its G block and X block are, with the part of x that is theirs, and whether the G block is another
        // than the slot's before
        int g_at[QW], x_at[QW];
        unsigned turns = 1;
#pragma unroll
        for (int q = 0; q < QW; ++q) {
            const int pos = q < w_n ? __builtin_amdgcn_readfirstlane((int)s_pos[w_lo + q]) : 0, r = pos >> 8, c = pos & 255;
            g_at[q] = r * C::BLOCK_BYTES | (r & 3) << 6;
            x_at[q] = C::X_PANEL | c * C::BLOCK_BYTES | (c & 3) << 6;
            if (q > 0 && g_at[q] != g_at[q - 1]) turns |= 1u << q;
        }

        f32x16 acc[QW];
#pragma unroll
        for (int q = 0; q < QW; ++q)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[q][v] = 0.f;

        constexpr int NU = TC / 16;   // 16-token matrix steps per chunk
        auto load_frag = [&](uint4 (&f)[NU], int at) {
#pragma unroll
            for (int u = 0; u < NU; ++u) f[u] = *reinterpret_cast<const uint4*>(smem + at + u * 1024);
        };

        if (q0 > 0) load_first();
#pragma unroll
        for (int d = 0; d < 8; ++d)
            if (d < 4 || whole) write_features(d >> 2, d & 3, 0);
#pragma unroll
        for (int k = 0; k < 8; ++k) load_row(k);
        load_next();
        for (int ci = 0; ci < nchunks; ++ci) {
            // chunk ci is in its buffer for every wave, and every wave is done reading chunk ci - 1
            lds_barrier();
            const int stage = (ci & 1) * C::STAGE, other = stage ^ C::STAGE;
            int read = read_at ^ stage;
            asm volatile("" : "+v"(read));   // (the addresses of all of a wave's blocks kept in vector registers spill)
            // The X fragment of block q + 1 is fetched before the products of block q are issued, that of G where it changes.  The
            // loop is unrolled: the two fragment sets alternate by name, not by copying.
            uint4 fa[2][NU], fb[NU];
            if (w_n > 0) load_frag(fa[0], read ^ x_at[0]);
#pragma unroll
            for (int q = 0; q < QW; ++q) {
                if (q < w_n) {
                    if (turns >> q & 1) load_frag(fb, read ^ g_at[q]);
                    if (q + 1 < QW) load_frag(fa[(q + 1) & 1], read ^ x_at[q + 1 < QW ? q + 1 : q]);
#pragma unroll
                    for (int u = 0; u < NU; ++u)
                        acc[q] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, fa[q & 1][u]),
                                                                         __builtin_bit_cast(bf16x8, fb[u]), acc[q], 0, 0, 0);
                }
                // this wave's share of chunk ci + 1, loaded during the chunk before, to its buffer; then that of chunk ci + 2 from memory
                if (q < 2 || ((q == 4 || q == 5) && whole)) {
                    write_features(q >> 2, (2 * q) & 3, other);
                    write_features(q >> 2, (2 * q + 1) & 3, other);
                }
                if (q == 2 || q == 3 || q == 6 || q == 7) {
                    load_row((q & 4) + 2 * (q & 1));
                    load_row((q & 4) + 2 * (q & 1) + 1);
                }
            }
            load_next();
            if (sum_mine && q0 == 0) {
                for (int t = sum_t0; t < TC / 8; t += sum_step) {
                    const int at = sum_place * C::BLOCK_BYTES + (t >> 1) * 1024 + (t & 1) * 512 +
                                   (((sum_f & 24) * 16 + (((sum_f & 7) ^ (sum_f >> 3)) << 4)) ^ (sum_place & 3) << 6);
                    const uint4 v = *reinterpret_cast<const uint4*>(smem + stage + at);
                    auto pair = [](uint32_t w) { return __uint_as_float(w << 16) + __uint_as_float(w & 0xffff0000u); };
                    sum += (pair(v.x) + pair(v.y)) + (pair(v.z) + pair(v.w));
                }
            }
        }
        lds_barrier();   // the next pass, or the sums of the bias, take the buffers
        if (sum_rows > 0 && q0 == 0) {
            float* s_sum = reinterpret_cast<float*>(smem);   // [sum_step][sum_width]
            if (sum_mine) s_sum[tid] = sum;
            lds_barrier();
            if (tid < sum_width) {
                float v = 0.f;
                for (int t = 0; t < sum_step; ++t) v += s_sum[t * sum_width + tid];
                const int row = s_rowid[sum_p0 + tid / 32];
                if (row >= 0) {
                    if (part) part[(size_t)a.nnz * 1024 + row * 32 + tid % 32] = v;
                    else static_cast<bf16_t*>(a.bias_out)[row * 32 + tid % 32] = Elem<bf16_t>::from_f32(v);
                }
            }
            lds_barrier();
        }

        // ---- store: result row j (X feature), column i (G feature) ----
#pragma unroll
        for (int q = 0; q < QW; ++q) {
            const int blk = q < w_n ? __builtin_amdgcn_readfirstlane(s_blk[w_lo + q]) : -1;
            if (blk >= 0) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const size_t o = (size_t)blk * 1024 + acc_row(v, h) * 32 + lrow;
                    // (partial sums are written once and read once, by sdd_reduce_kernel: stored and loaded non-temporally
                    // they leave the operands of the next product in the last-level cache)
                    if (part) __builtin_nontemporal_store(acc[q][v], part + o);
                    else out[o] = Elem<bf16_t>::from_f32(acc[q][v]);
                }
            }
        }
    }
}

template <bool BIAS>
__global__ __launch_bounds__(512) void sdd_bf16_kernel(SddArgs a) {
    if (a.rows == 8) sdd_rectangle<BIAS, 8>(a);
    else sdd_rectangle<BIAS, 16>(a);
}

}  // namespace pbs
