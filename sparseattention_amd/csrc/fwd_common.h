// Helpers shared by the forward kernels: register types, per-dtype MFMA wrappers, the direct global->LDS
// load, the LDS row swizzles and the constants of the online softmax.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "kernels.h"

namespace sa {
namespace {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

#define SA_LDS __attribute__((address_space(3)))

template <int DT>
struct Elem;

template <>
struct Elem<0> {  // bf16
    static __device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
    }
    // 16x16x32 product; lane l supplies row/column l%16 and the 8 contraction indices 8*(l/16)..+7, and
    // receives column l%16, rows 4*(l/16)..+3
    static __device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                       0, 0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
        const f32x2 f = {lo, hi};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
    }
    static __device__ __forceinline__ uint32_t scale2(uint32_t w, float s) {  // both halves times s, rounded again
        return pack2(__uint_as_float(w << 16) * s, __uint_as_float(w & 0xffff0000u) * s);
    }
    template <class P>
    static __device__ __forceinline__ u32x2 tr_read(P lds_ptr) {
        return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4bf16((SA_LDS bf16x4 *)lds_ptr));
    }
    static __device__ __forceinline__ u32x4 ones4() {  // eight 1.0 values, an all-ones MFMA operand
        return u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
    }
};

template <>
struct Elem<1> {  // fp16
    static __device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                      0, 0);
    }
    static __device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                      0, 0);
    }
    static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
        const f32x2 f = {lo, hi};
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, f16x2));
    }
    static __device__ __forceinline__ uint32_t scale2(uint32_t w, float s) {
        const f16x2 h = __builtin_bit_cast(f16x2, w);
        return pack2((float)h.x * s, (float)h.y * s);
    }
    template <class P>
    static __device__ __forceinline__ u32x2 tr_read(P lds_ptr) {
        // the transposing read only moves 16-bit lanes around, so the bf16 flavour serves fp16 too
        return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4bf16((SA_LDS bf16x4 *)lds_ptr));
    }
    static __device__ __forceinline__ u32x4 ones4() {
        return u32x4{0x3c003c00u, 0x3c003c00u, 0x3c003c00u, 0x3c003c00u};
    }
};

// Exchange a value between lane and lane^32 and combine: returns op(x[lane], x[lane^32]) in all lanes.
__device__ __forceinline__ float half_swap_max(float x) {
    const uint32_t u = __float_as_uint(x);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

constexpr float kNegInf = -__builtin_inff();

// 16 bytes per lane from global memory (wave-uniform base + per-lane byte offset) straight into LDS:
// lane i of the wave writes LDS address lds_addr + 16*i.
// Issued through inline assembly on purpose: the compiler then does not track it, so it does not hold
// back later LDS reads of the OTHER buffer until the transfer lands.  Whoever reads the destination
// must execute "s_waitcnt vmcnt(0)" and a workgroup barrier first (the main loop does).
// The load takes its LDS address from m0, which needs a wait state after a scalar write.  The write of m0 and the
// s_nop therefore stay INSIDE this asm statement: handing the address over as an "{m0}" input leaves the copy into
// the (reserved) register to the compiler, with no guarantee of the wait state or that two loads do not share one
// copy, and a build of that form ended in a GPU memory fault.
// STREAM: the bytes are read once by the whole launch (the K/V rows of the few-rows kernels): the load carries the
// non-temporal hint, with which a streaming read runs at 7.1 TB/s on this device against 6.3 TB/s without.
// DEVICE: what another workgroup of this launch has handed over (HandOver).
template <bool STREAM = false, bool DEVICE = false>
__device__ __forceinline__ void dma16(const void *base, uint32_t lane_offset, uint32_t lds_addr) {
    // the base is wave-uniform by construction; say so in a way the register allocator cannot miss
    const uint64_t b = (uint64_t)(uintptr_t)base;
    // (readfirstlane returns a signed int: widen through uint32_t, or the low half sign-extends)
    const uint64_t ub = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b) |
                        ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) << 32);
    lds_addr = __builtin_amdgcn_readfirstlane(lds_addr);
    if constexpr (DEVICE) {
        asm volatile(
            "s_mov_b32 m0, %2\n\t"
            "s_nop 0\n\t"
            "global_load_lds_dwordx4 %0, %1 sc1"
            :
            : "v"(lane_offset), "s"(ub), "s"(lds_addr)
            : "memory");
    } else if constexpr (STREAM) {
        asm volatile(
            "s_mov_b32 m0, %2\n\t"
            "s_nop 0\n\t"
            "global_load_lds_dwordx4 %0, %1 nt"
            :
            : "v"(lane_offset), "s"(ub), "s"(lds_addr)
            : "memory");
    } else {
        asm volatile(
            "s_mov_b32 m0, %2\n\t"
            "s_nop 0\n\t"
            "global_load_lds_dwordx4 %0, %1"
            :
            : "v"(lane_offset), "s"(ub), "s"(lds_addr)
            : "memory");  // m0 is written; nothing else in these kernels keeps a value in it
    }
}

// The same with an address per lane.
__device__ __forceinline__ void dma16_lane(const void *lane_addr, uint32_t lds_addr) {
    lds_addr = __builtin_amdgcn_readfirstlane(lds_addr);
    asm volatile(
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %0, off"
        :
        : "v"(lane_addr), "s"(lds_addr)
        : "memory");
}

// 4 bytes per lane: lane i of the wave writes LDS address lds_addr + 4*i.
__device__ __forceinline__ void dma4(const void *base, uint32_t lane_offset, uint32_t lds_addr) {
    const uint64_t b = (uint64_t)(uintptr_t)base;
    const uint64_t ub = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b) |
                        ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) << 32);
    lds_addr = __builtin_amdgcn_readfirstlane(lds_addr);
    asm volatile(
        "s_mov_b32 m0, %2\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dword %0, %1"
        :
        : "v"(lane_offset), "s"(ub), "s"(lds_addr)
        : "memory");
}
__device__ __forceinline__ void dma4_lane(const void *lane_addr, uint32_t lds_addr) {
    lds_addr = __builtin_amdgcn_readfirstlane(lds_addr);
    asm volatile(
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dword %0, off"
        :
        : "v"(lane_addr), "s"(lds_addr)
        : "memory");
}

// What a lane whose 16 bytes do not exist fetches.
__device__ const uint32_t kZeros[4] __attribute__((aligned(16))) = {0u, 0u, 0u, 0u};

// N dwords from N wave-uniform addresses by scalar loads that are issued back to back and share ONE wait.  Left to
// the compiler, loads whose addresses it forms one after the other are waited for one after the other as well, a
// memory round trip each; at the start of a Q tile that is most of the time before the first K/V request.
template <int N>
__device__ __forceinline__ void scalar_gather(const int32_t *const (&a)[N], int (&o)[N]) {
    static_assert(N == 2 || N == 4 || N == 6 || N == 8 || N == 10,
                  "counts, first slots of both lists for 1, 2 or 4 entries per chunk, or both");
    const uint64_t *const q = reinterpret_cast<const uint64_t *>(&a[0]);  // (pointers as 64-bit scalars)
    if constexpr (N == 2) {
        asm volatile(
            "s_load_dword %0, %2, 0x0\n\ts_load_dword %1, %3, 0x0\n\ts_waitcnt lgkmcnt(0)"
            : "=&s"(o[0]), "=&s"(o[1])
            : "s"(q[0]), "s"(q[1])
            : "memory");
    } else if constexpr (N == 8) {
        asm volatile(
            "s_load_dword %0, %8, 0x0\n\ts_load_dword %1, %9, 0x0\n\ts_load_dword %2, %10, 0x0\n\t"
            "s_load_dword %3, %11, 0x0\n\ts_load_dword %4, %12, 0x0\n\ts_load_dword %5, %13, 0x0\n\t"
            "s_load_dword %6, %14, 0x0\n\ts_load_dword %7, %15, 0x0\n\ts_waitcnt lgkmcnt(0)"
            : "=&s"(o[0]), "=&s"(o[1]), "=&s"(o[2]), "=&s"(o[3]), "=&s"(o[4]), "=&s"(o[5]), "=&s"(o[6]), "=&s"(o[7])
            : "s"(q[0]), "s"(q[1]), "s"(q[2]), "s"(q[3]), "s"(q[4]), "s"(q[5]), "s"(q[6]), "s"(q[7])
            : "memory");
    } else if constexpr (N == 4) {
        asm volatile(
            "s_load_dword %0, %4, 0x0\n\ts_load_dword %1, %5, 0x0\n\ts_load_dword %2, %6, 0x0\n\t"
            "s_load_dword %3, %7, 0x0\n\ts_waitcnt lgkmcnt(0)"
            : "=&s"(o[0]), "=&s"(o[1]), "=&s"(o[2]), "=&s"(o[3])
            : "s"(q[0]), "s"(q[1]), "s"(q[2]), "s"(q[3])
            : "memory");
    } else if constexpr (N == 6) {
        asm volatile(
            "s_load_dword %0, %6, 0x0\n\ts_load_dword %1, %7, 0x0\n\ts_load_dword %2, %8, 0x0\n\t"
            "s_load_dword %3, %9, 0x0\n\ts_load_dword %4, %10, 0x0\n\ts_load_dword %5, %11, 0x0\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&s"(o[0]), "=&s"(o[1]), "=&s"(o[2]), "=&s"(o[3]), "=&s"(o[4]), "=&s"(o[5])
            : "s"(q[0]), "s"(q[1]), "s"(q[2]), "s"(q[3]), "s"(q[4]), "s"(q[5])
            : "memory");
    } else {
        asm volatile(
            "s_load_dword %0, %10, 0x0\n\ts_load_dword %1, %11, 0x0\n\ts_load_dword %2, %12, 0x0\n\t"
            "s_load_dword %3, %13, 0x0\n\ts_load_dword %4, %14, 0x0\n\ts_load_dword %5, %15, 0x0\n\t"
            "s_load_dword %6, %16, 0x0\n\ts_load_dword %7, %17, 0x0\n\ts_load_dword %8, %18, 0x0\n\t"
            "s_load_dword %9, %19, 0x0\n\ts_waitcnt lgkmcnt(0)"
            : "=&s"(o[0]), "=&s"(o[1]), "=&s"(o[2]), "=&s"(o[3]), "=&s"(o[4]), "=&s"(o[5]), "=&s"(o[6]), "=&s"(o[7]),
              "=&s"(o[8]), "=&s"(o[9])
            : "s"(q[0]), "s"(q[1]), "s"(q[2]), "s"(q[3]), "s"(q[4]), "s"(q[5]), "s"(q[6]), "s"(q[7]), "s"(q[8]), "s"(q[9])
            : "memory");
    }
}

// Swizzles of the 16-byte pieces inside an LDS row.  Rows are stored unpadded (D*2 bytes) because a
// direct global->LDS load writes 64 lanes x 16 bytes contiguously; instead the piece index is XORed
// with a function of the row so that
//   K: the 16 rows read together by one quarter-wave ds_read_b128 fall into 16 different bank groups,
//   V: the 4 rows touched by one half-wave transposing read fall into 4 different 64-byte bank groups.
template <int D>
__device__ __forceinline__ int k_swizzle(int row) {
    return D >= 128 ? (row & 15) : ((row >> 1) & 7);
}
template <int D>
__device__ __forceinline__ int v_swizzle(int row) {
    return D >= 128 ? 4 * (row & 3) : 4 * ((row >> 1) & 1);
}

// Several workgroups leave parts of one result in memory; the last of them to arrive adds the parts up, in the same launch.
// What one workgroup hands to another goes by stores and loads of device scope (sc1): they pass the L2 of their XCD by, so
// nothing has to be written back or invalidated there, where other workgroups keep their operands (a release and an
// acquire of device scope take 5.6 us of a workgroup, the counter alone 0.4).  512 workgroups, parts of 8 KiB of which four meet: stores
// 1.6 us (0.9 where the four run on one XCD), counter 0.4, loads 1.2 ... 1.6.
constexpr int kDeviceScope = 16;  // (the sc1 bit of a buffer instruction's modifiers)
struct HandOver {
    __amdgpu_buffer_rsrc_t rsrc;
    // `bytes` (less than 2 GiB) from a wave-uniform base; accesses outside them do nothing
    __device__ __forceinline__ HandOver(void *base, uint32_t bytes) {
        const uint64_t b = (uint64_t)(uintptr_t)base;
        const uint64_t ub = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b) |
                            ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) << 32);
        rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(uintptr_t)ub, 0, (int)bytes, 0x00027000);
    }
    __device__ __forceinline__ void put(uint32_t at, f32x4 x) const {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), rsrc, (int)at, 0, kDeviceScope);
    }
    __device__ __forceinline__ void put(uint32_t at, f32x2 x) const {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), rsrc, (int)at, 0, kDeviceScope);
    }
    __device__ __forceinline__ f32x4 get4(uint32_t at) const {
        return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)at, 0, kDeviceScope));
    }
    __device__ __forceinline__ f32x2 get2(uint32_t at) const {
        return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, (int)at, 0, kDeviceScope));
    }
};
// One thread of each of n <= kArrivalMost workgroups, after what the workgroup hands over has been stored (every wave: vmcnt(0),
// then a barrier): true for the last one.  The word needs no first value: its upper 56 bits are the launch's number
// (next_launch_tag, no two launches of a process share one), its low 8 bits count.  A word with other upper bits, whatever the memory held, counts
// as zero.  The last one leaves zero, so that a replay of a captured launch, which brings the same number, finds no count.
constexpr int kArrivalMost = 255;
__device__ __forceinline__ bool arrives_last(uint64_t *word, uint64_t tag, int n) {
    uint64_t old = __hip_atomic_fetch_add(word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((old & ~0xffull) != tag) {
        // (the count was added to what the memory held: harmless, and never more than n times)
        uint64_t seen = old + 1;
        for (;;) {
            if ((seen & ~0xffull) == tag) {  // another one has put the number there meanwhile
                old = __hip_atomic_fetch_add(word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
            if (__hip_atomic_compare_exchange_strong(word, &seen, tag | 1ull, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                old = tag;
                break;
            }
        }
    }
    if ((int)(old & 0xff) + 1 != n) return false;
    __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// The same without a common word, whose atomics go through one place one after the other (0.5 us each: seven workgroups 3.4 us, this
// way 1.2): each of n <= 64 workgroups has a word of its own.  One wave of each, after what its workgroup hands over has been stored: it
// sets its word to the launch's number, waits until that is in memory and looks at all n.  Whoever's word gets there last sees all set, so at
// least one workgroup is told true; more than one may be, and then each does the same work and leaves the same bits.  Who
// is told true clears the words (all have been set then), so that a replay of a captured launch, which brings the same number, finds none.
__device__ __forceinline__ bool all_arrived(uint64_t *words, uint64_t tag, int mine, int n) {
    const int lane = threadIdx.x & 63;
    const HandOver h(words, 8u * (uint32_t)n);
    const u32x2 set = {(uint32_t)tag, (uint32_t)(tag >> 32)};
    if (lane == 0) h.put(8u * (uint32_t)mine, __builtin_bit_cast(f32x2, set));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const u32x2 seen = __builtin_bit_cast(u32x2, h.get2(8u * (uint32_t)min(lane, n - 1)));
    const bool all = __builtin_amdgcn_ballot_w64(seen.x == set.x && seen.y == set.y) == ~0ull;
    if (all && lane < n) h.put(8u * (uint32_t)lane, f32x2{0.f, 0.f});
    return all;
}

// Whether the workgroup of this word has handed over what it has.  One wave.
__device__ __forceinline__ bool other_arrived(uint64_t *words, uint64_t tag, int other) {
    const HandOver h(words, 8u * (uint32_t)(other + 1));
    const u32x2 seen = __builtin_bit_cast(u32x2, h.get2(8u * (uint32_t)other));
    return __builtin_amdgcn_readfirstlane(seen.x == (uint32_t)tag && seen.y == (uint32_t)(tag >> 32));
}

// The sum of n parts that workgroups have handed over: this wave's N blocks of 32 x 32 values, 16 a lane, the lane's four of run g of a
// block at rows_at + part * rows_step + 1024 (4 block + g) (where a wave leaves its accumulators, 1 KiB a store), with reference value
// (-inf: no attended key) and sum of the lane's row at state_at + part * state_step.  In the order of the parts, whoever adds.  The
// first B parts are under way while the largest reference value is looked for, by fours: one round trip for up to four parts, one more for every four
// beyond them and for every B parts behind the first B.
template <int N, int B>
__device__ __forceinline__ void add_parts(const HandOver &rows, uint32_t rows_at, uint32_t rows_step, const HandOver &state, uint32_t state_at,
                                          uint32_t state_step, int n, f32x16 (&acc)[N], float &M, float &L) {
    f32x4 x[B][4 * N];
    f32x2 st[B];
    auto request = [&](int i0) {
#pragma unroll
        for (int i = 0; i < B; i++) {
            const uint32_t part = (uint32_t)min(i0 + i, n - 1);  // (past the last one: that one again, left out below)
            st[i] = state.get2(state_at + part * state_step);
#pragma unroll
            for (int g = 0; g < 4 * N; g++) x[i][g] = rows.get4(rows_at + part * rows_step + 1024u * g);
        }
    };
    request(0);
    float m = kNegInf;
    for (int i0 = 0; i0 < n; i0 += 4) {
        f32x2 s4[4];
#pragma unroll
        for (int i = 0; i < 4; i++) s4[i] = state.get2(state_at + (uint32_t)min(i0 + i, n - 1) * state_step);
#pragma unroll
        for (int i = 0; i < 4; i++) m = fmaxf(m, s4[i].x);
    }
    M = m;
    L = 0.f;
    const float M0 = m == kNegInf ? 0.f : m;  // (no part saw an attended key: every weight is 0)
#pragma unroll
    for (int d = 0; d < N; d++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[d][e] = 0.f;
#pragma unroll 1
    for (int i0 = 0;;) {
#pragma unroll
        for (int i = 0; i < B; i++) {
            if (i0 + i >= n) break;
            const float w = __builtin_amdgcn_exp2f(st[i].x - M0);
            L = __builtin_fmaf(w, st[i].y, L);
#pragma unroll
            for (int g = 0; g < 4 * N; g++)
#pragma unroll
                for (int e = 0; e < 4; e++) acc[g / 4][4 * (g % 4) + e] = __builtin_fmaf(w, x[i][g][e], acc[g / 4][4 * (g % 4) + e]);
        }
        i0 += B;
        if (i0 >= n) break;
        request(i0);
    }
}

// log2-domain slack before the running maximum is raised (and the accumulator rescaled).  Scores are
// exponentiated against a reference value that may lag the true row maximum by up to this much, so
// P stays <= 2^kMaxSlack; the final division by the row sum cancels the reference exactly.
constexpr float kMaxSlack = 8.0f;

// List entries kept in LDS per Q tile (8 KiB); longer lists are read from global memory per chunk.
constexpr int kListCap = 2048;
// Persistent workgroups keep two lists in the same space, of the Q tile at hand and of the next one.
constexpr int kPsListCap = 1024;

template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {  // f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>)
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

// Raises a kernel's dynamic shared-memory limit to `bytes`, once per device: `done` is the caller's bit mask of the
// devices (ordinals below 64) that have it.  Two threads racing here set the same value twice.
template <class K>
hipError_t allow_dynamic_smem(K kern, int bytes, unsigned long long &done) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const unsigned long long bit = dev >= 0 && dev < 64 ? 1ull << dev : 0ull;
    if (bit != 0 && (__atomic_load_n(&done, __ATOMIC_RELAXED) & bit)) return hipSuccess;
    e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess && bit != 0) __atomic_fetch_or(&done, bit, __ATOMIC_RELAXED);
    return e;
}

}  // namespace
}  // namespace sa
