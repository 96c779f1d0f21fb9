// Shared device helpers for the gfx950 block-sparse kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pbs {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

struct bf16_t {
    uint16_t bits;
};

// Per element type: bytes, and the conversions from and to float.
template <typename T>
struct Elem;

template <>
struct Elem<float> {
    static constexpr int ESZ = 4;
    static __device__ __forceinline__ float from_f32(float v) { return v; }
    static __device__ __forceinline__ float to_f32(float v) { return v; }
};

template <>
struct Elem<bf16_t> {
    static constexpr int ESZ = 2;
    // round to nearest even, NaN kept quiet: the hardware conversion (v_cvt_pk_bf16_f32, two values per
    // instruction where the compiler can pair them)
    static __device__ __forceinline__ bf16_t from_f32(float v) {
        bf16_t r;
        r.bits = __builtin_bit_cast(uint16_t, static_cast<__bf16>(v));
        return r;
    }
    static __device__ __forceinline__ float to_f32(bf16_t v) { return __uint_as_float(((uint32_t)v.bits) << 16); }
};

// Row of accumulator register v (0..15) held by a lane of half h in a 32x32 MFMA result;
// the column is (lane & 31).
static __device__ __forceinline__ int acc_row(int v, int h) { return 8 * (v >> 2) + 4 * h + (v & 3); }

// A row/column pointer value read from a caller's index array, forced into [0, nnz]: a corrupt
// pointer array then selects wrong entries instead of reading outside the entry list.
static __device__ __forceinline__ int clamp_entry(int v, int nnz) { return v < 0 ? 0 : (v > nnz ? nnz : v); }

// ds_read_b64_tr_b16: within each group of 16 lanes, lane s passes the LDS address of 4 consecutive
// 16-bit elements (row s/4 of a 4 x 16 tile, columns 4*(s%4)..+3) and lane j receives column j of
// the tile: the 4 rows' elements, in row order.
static __device__ __forceinline__ uint2 tr16_b64(const unsigned char* lds_ptr) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(lds_ptr));
    return __builtin_bit_cast(uint2, v);
}

// Volatile accesses to LDS words other waves write or poll.  The pointer is cast to the LDS address
// space explicitly: a volatile access through a generic pointer is compiled to a flat instruction,
// which takes the long way round through the vector memory path.
typedef int __attribute__((address_space(3))) lds_int;
static __device__ __forceinline__ int lds_peek(const int* p) { return *(const volatile lds_int*)p; }
static __device__ __forceinline__ void lds_poke(int* p, int v) { *(volatile lds_int*)p = v; }

// the lane's number, made where it is asked for: it needs no register until then
static __device__ __forceinline__ int lane_now() {
    int lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(lane));
    return lane;
}

// Waits of the barrier-free kernels that ran into their bound, counted over the life of the process (one word per
// GPU).  Such a wait means a broken progress protocol; the kernel also turns the affected results into NaN.
static __device__ unsigned g_protocol_failures;
static __device__ __forceinline__ void count_protocol_failure() {
    if (lane_now() == 0) atomicAdd(&g_protocol_failures, 1u);
}

// a wave-uniform pointer, forced into scalar registers
static __device__ __forceinline__ const unsigned char* uniform_ptr(const unsigned char* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return reinterpret_cast<const unsigned char*>(((uint64_t)hi << 32) | lo);
}

// one DMA instruction: lane p copies the 16 bytes at base + voff to LDS chunk (lds_base/16 + p).
// M0 is written inside the statement and cannot be named as a clobber (the compiler treats it as a
// reserved register and rejects that with a warning about undefined behaviour); these kernels contain
// nothing else that makes the compiler use M0 (no LDS-DMA builtins, no dynamically indexed registers).
static __device__ __forceinline__ void dma16(unsigned lds_base_uniform, const unsigned char* base_uniform, unsigned voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\t"
                 :
                 : "s"(lds_base_uniform), "v"(voff), "s"(base_uniform)
                 : "memory");
}

// the same with an address per lane
static __device__ __forceinline__ void dma16_lanes(unsigned lds_base_uniform, const unsigned char* at) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\t"
                 :
                 : "s"(lds_base_uniform), "v"(at)
                 : "memory");
}

// 16 bytes per lane from `off` on in a buffer of `bytes` bytes (both below 2^31; base and bytes wave-uniform); zeros, and no memory
// access, where off lies behind its end
static __device__ __forceinline__ uint4 buffer16(const unsigned char* base_uniform, unsigned bytes, unsigned off) {
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(base_uniform), 0, bytes, 0x00020000);
    return __builtin_bit_cast(uint4, (u32x4)__builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0));
}

// A buffer of `bytes` bytes (below 2^32) at a wave-uniform address, and the same from `voff` on in it: lanes whose 16 bytes lie behind its end
// read nothing and put zeros in the LDS.  (All of an offset is in voff: what the instruction adds from a scalar register is no part of
// its check.)
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
static __device__ __forceinline__ u32x4_t bounded_buffer(const unsigned char* base_uniform, unsigned bytes) {
    const uint64_t at = reinterpret_cast<uint64_t>(base_uniform);
    return u32x4_t{(unsigned)__builtin_amdgcn_readfirstlane((uint32_t)at), (unsigned)__builtin_amdgcn_readfirstlane((uint32_t)(at >> 32)),
                   (unsigned)__builtin_amdgcn_readfirstlane(bytes), 0x00020000u};
}
static __device__ __forceinline__ void dma16_bounded(unsigned lds_base_uniform, u32x4_t buffer, unsigned voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds\n\t"
                 :
                 : "s"(lds_base_uniform), "v"(voff), "s"(buffer)
                 : "memory");
}

// the 4-byte form: lane p copies the 4 bytes at base + voff to LDS word (lds_base/4 + p)
static __device__ __forceinline__ void dma4(unsigned lds_base_uniform, const unsigned char* base_uniform, unsigned voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2\n\t"
                 :
                 : "s"(lds_base_uniform), "v"(voff), "s"(base_uniform)
                 : "memory");
}
// wait until at most n (wave-uniform) of this wave's DMA loads are outstanding.  Loads retire in order, so a smaller n than necessary is only slower, never wrong.
// n is a constant, or one of two (one branch): the branches over all counts, with one that a loop works out, cost a third of a kernel's time.
static __device__ __forceinline__ void wait_dma(int n) {
#define PBS_W(N) case N: asm volatile("s_waitcnt vmcnt(" #N ")" ::: "memory"); break;
    switch (n) {
        PBS_W(0) PBS_W(1) PBS_W(2) PBS_W(3) PBS_W(4) PBS_W(5) PBS_W(6) PBS_W(7) PBS_W(8)
        PBS_W(9) PBS_W(10) PBS_W(11) PBS_W(12) PBS_W(13) PBS_W(14) PBS_W(15) PBS_W(16)
        PBS_W(17) PBS_W(18) PBS_W(19) PBS_W(20) PBS_W(21) PBS_W(22) PBS_W(23) PBS_W(24)
        PBS_W(25) PBS_W(26) PBS_W(27) PBS_W(28) PBS_W(29) PBS_W(30) PBS_W(31) PBS_W(32)
        PBS_W(33) PBS_W(34) PBS_W(35) PBS_W(36) PBS_W(37) PBS_W(38) PBS_W(39) PBS_W(40)
        PBS_W(41) PBS_W(42) PBS_W(43) PBS_W(44) PBS_W(45) PBS_W(46) PBS_W(47) PBS_W(48)
        default: asm volatile("s_waitcnt vmcnt(48)" ::: "memory"); break;
    }
#undef PBS_W
}
// barrier of a wave that has no DMA in flight or does not care (its LDS accesses complete first)
static __device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
static __device__ __forceinline__ void drain_barrier() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

static constexpr int NUM_XCD = 8;

// Workgroups are handed to the 8 XCDs round-robin by id.  Give each XCD one contiguous range of
// logical tile ids, walked in launch order, so tiles that share an operand panel run on the same
// XCD (one L2) at about the same time.  Returns -1 for the padding ids of the last range.
static __device__ __forceinline__ int xcd_tile_id(int wg, int total) {
    const int per = (total + NUM_XCD - 1) / NUM_XCD;
    const int id = (wg % NUM_XCD) * per + wg / NUM_XCD;
    return id < total ? id : -1;
}
static inline int xcd_grid(int total) { return ((total + NUM_XCD - 1) / NUM_XCD) * NUM_XCD; }

// Persistent workgroups of `streams` token streams x `groups` column groups, at most one for each of the 256 CUs: `sets` (1 or 2) sets of the groups, each dealt
// stream by stream in equal runs to every sets-th XCD, so no XCD gets more than it has CUs.  (With whole streams to an XCD, 7 groups and 36 streams made 35
// workgroups on 32 CUs: three of them, and with them the launch, began when the others had ended.  254 such products of the column kernel are 1.16 times as fast, 177 of the
// wide kernel 1.35 times; where whole streams fit, these kernels are level, 1.002 and 1.005 times as fast in whole streams in 200 and 80 products.)  The streams are numbered in steps of `step`, which has no
// factor in common with their number: where the first ones have a tile more than the others (`tiles` of them in all), they are so on all XCDs (2560 -> 2560 density 0.5,
// 9000 tokens 99 -> 95 us; where all have as many, 4096 -> 4096 at 16384 tokens, any step but 1 takes 0.8 % more).
static inline unsigned stream_grid_blocks(int streams, int groups, int sets) {
    const int parts = NUM_XCD / sets;
    return (unsigned)(NUM_XCD * (((long long)(groups / sets) * streams + parts - 1) / parts));
}
static inline int stream_step(int streams, int tiles) {
    if (tiles % streams == 0) return 1;
    auto shared = [&](int a) {
        int b = streams;
        while (b) {
            const int r = a % b;
            a = b;
            b = r;
        }
        return a > 1;
    };
    int step = (int)(0.618 * streams) + 1;   // (the golden section: any run of streams is spread evenly)
    while (shared(step)) ++step;
    return step;
}
static __device__ __forceinline__ bool stream_and_group(int wg, int streams, int step, int groups, int sets, int& stream, int& group) {
    const int x = wg % NUM_XCD, gs = groups / sets, part = x / sets, parts = NUM_XCD / sets;
    const int lo = (int)((long long)gs * streams * part / parts), hi = (int)((long long)gs * streams * (part + 1) / parts);
    const int at = lo + wg / NUM_XCD, i = at / gs;
    stream = (int)((long long)i * step % streams);
    group = x % sets * gs + at - i * gs;
    return at < hi;
}

}  // namespace pbs
