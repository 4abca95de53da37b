// Vector types and small device helpers of the attention kernels that work on the matrix cores (attention_fast.hip,
// attention_prefill.hip).
#pragma once
#include "attention_common.h"

namespace hqmq {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef const uint2 __attribute__((address_space(3))) *lds_u2_ptr;
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
typedef uint4v uint4v_a8 __attribute__((aligned(8)));         // a 16-byte vector at an 8-byte aligned address
typedef uint32_t uint32_a2 __attribute__((aligned(2)));       // a dword at a 2-byte aligned address

template <int DT>
__device__ __forceinline__ half4 chunk_to_half(uint2 w) {
    if (DT == HQMQ_F16) return __builtin_bit_cast(half4, w);
    half4 r;
    r[0] = (_Float16)__uint_as_float(w.x << 16); r[1] = (_Float16)__uint_as_float(w.x & 0xffff0000u);
    r[2] = (_Float16)__uint_as_float(w.y << 16); r[3] = (_Float16)__uint_as_float(w.y & 0xffff0000u);
    return r;
}

// Two codewords (16 bytes) of a table in the cache dtype -> the same two as fp16
template <int DT>
__device__ __forceinline__ uint4v pair_to_half(uint4v w) {
    if (DT == HQMQ_F16) return w;
    const uint2 a = __builtin_bit_cast(uint2, chunk_to_half<DT>(uint2{w[0], w[1]}));
    const uint2 b = __builtin_bit_cast(uint2, chunk_to_half<DT>(uint2{w[2], w[3]}));
    return uint4v{a.x, a.y, b.x, b.y};
}

// One word of a caller's array that no kernel writes while this one runs, at a wave-uniform index: read through the
// constant address space, i.e. by a scalar load.  (As a vector load it is followed by a wait for every vector load
// before it: in the prologues below, for the table loads, and once per dependent word.)
__device__ __forceinline__ int32_t uniform_word(const int32_t *a, int64_t i) {
    typedef const int32_t __attribute__((address_space(4))) *const_i32_ptr;
    return ((const_i32_ptr)(uintptr_t)a)[i];
}

// acc * scale[hi] (+ add): for fp16 scales one mixed-precision fma reads the half directly
template <int DT>
__device__ __forceinline__ float scaled(float acc, uint32_t pair, int hi, float add) {
    if (DT == HQMQ_F16) return __builtin_fmaf(acc, (float)__builtin_bit_cast(half2v, pair)[hi], add);
    return __builtin_fmaf(acc, __uint_as_float(hi ? (pair & 0xffff0000u) : (pair << 16)), add);
}
// Four weights times the scales of their tokens, each product rounded to fp16 once: for fp16 scales one mixed-precision fma a weight,
// no more than the conversions and packed products that rounded the weight first and the product again.
template <int DT>
__device__ __forceinline__ half4 weigh(const float (&w)[4], uint2 scales) {
    half4 r;
#pragma unroll
    for (int e = 0; e < 4; e++) r[e] = (_Float16)scaled<DT>(w[e], e < 2 ? scales.x : scales.y, e & 1, 0.f);
    return r;
}

typedef const uint4v __attribute__((address_space(3))) *lds_u4_ptr;
typedef const uint32_t __attribute__((address_space(3))) *lds_u1_ptr;

// x / d through the multiplier the host worked out for d (m = ceil(2^32 / d), exact while x * d < 2^32; m = 0 stands for
// d = 1: the launcher keeps these kernels for launches where every divisor has its multiplier, see launch_layout).
// No division as a fall-back: its expansion, once per use, made the prologue a chain of branches, each with its own
// re-read of the argument block and a wait for it.
__device__ __forceinline__ unsigned fast_div(unsigned x, unsigned d, unsigned m) { return m ? __umulhi(x, m) : x; }

__device__ __forceinline__ half8 cat8(half4 x, half4 y) { return __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7); }

// The parameter block spans several 64-byte lines of the kernel-argument segment, and the prologue reads them one
// after the other as its address arithmetic proceeds: every first touch of a line is a miss of the scalar cache
// that the next scalar load waits behind.  One dword of every line, requested together at the very start, turns
// the chain of misses into one.
__device__ __forceinline__ void touch_kernargs() {
    typedef const uint32_t __attribute__((address_space(4))) *karg_ptr;
    karg_ptr ka = (karg_ptr)__builtin_amdgcn_kernarg_segment_ptr();
    uint32_t t = 0;
#pragma unroll
    for (int i = 0; i < (int)((sizeof(AttnParams) + 63) / 64); i++) t |= ka[16 * i];
    asm volatile("" ::"s"(t));
}

// Loads that land in LDS.  The compiler neither sees nor counts them; loads come back in the order they were requested, so vmcnt(n) with n
// no more than the loads requested after them waits for them, and so does the use of a register loaded after them.
template <int N>
__device__ __forceinline__ void wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ __forceinline__ const uint8_t *uniform_ptr(const uint8_t *p) {
    const uint64_t v = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (const uint8_t *)(((uint64_t)hi << 32) | lo);
}
// 64 lanes x 16 bytes from base + voff (+ the instruction's offset, which counts for both sides) to LDS at m0 + 16 * lane.  Between a
// write of m0 and the load that reads it the hardware asks for one wait state; the compiler, which inserts it elsewhere, does not look
// inside an asm block.
__device__ __forceinline__ void lds_load16(uint32_t lds_base, const uint8_t *base, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_base), "v"(voff), "s"(base) : "memory");
}
// The K and V codeword tables in 1 KB units dealt to the wavefronts round-robin, straight to their places in LDS (whole units: the last
// pair of codewords again past a table's end).
template <int WV>
__device__ __forceinline__ void land_tables(const uint8_t *k, uint32_t kbytes, const uint8_t *v, uint32_t vbytes, uint32_t k_at, uint32_t v_at, int wave, int lane) {
    const int ku = (int)((kbytes + 1023u) >> 10), nu = ku + (int)((vbytes + 1023u) >> 10);
    for (int u = wave; u < nu; u += WV) {
        const bool isv = u >= ku;
        const uint32_t uu = (uint32_t)(isv ? u - ku : u);
        const uint32_t off = min(uu * 1024u + (uint32_t)lane * 16u, (isv ? vbytes : kbytes) - 16u);
        lds_load16((isv ? v_at : k_at) + uu * 1024u, isv ? v : k, off);
    }
}

}  // namespace hqmq
