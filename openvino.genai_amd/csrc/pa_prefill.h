// What the matrix kernels of a step's chunks share (pa_prefill16.hip, pa_prefill_dense.hip): matrix and lane-swap
// instructions, conversions, copies into LDS and the waits that go with them.
#pragma once
#include "pa_device.h"

namespace pa {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef short s8v __attribute__((ext_vector_type(8)));
typedef short s4v __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

constexpr int TOK = 32;
constexpr float LOG2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;

template <int DT>
__device__ __forceinline__ f4 mma(const s8v& a, const s8v& b, const f4& c) {
    if (DT == DT_F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a), __builtin_bit_cast(h8, b), c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, a), __builtin_bit_cast(b8, b), c, 0, 0, 0);
}

__device__ __forceinline__ s4v lds_read_tr16(const uint8_t* p) {
    typedef s4v __attribute__((address_space(3))) * lds_ptr;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)p);
}

// Reductions over the four 16-lane groups of a wave with the gfx950 lane-swap instructions (no LDS round trip):
// v_permlane16_swap exchanges the odd 16-lane rows of its first operand with the even rows of the second,
// v_permlane32_swap the upper half of the first with the lower half of the second.  With both operands holding
// the same value the pair afterwards holds, per lane, the values of the two rows (halves) being combined.
__device__ __forceinline__ void swap_rows16(float& a, float& b) {
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ void swap_halves32(float& a, float& b) {
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
// (the maxima as instructions of their own: behind the lane swaps the compiler no longer knows its operands to be
// ordinary numbers and puts a quieting `v_max x, x, x` in front of every fmaxf)
__device__ __forceinline__ float max_raw(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float xor_max_g(float v) {
    float a = v, b = v;
    swap_rows16(a, b);
    a = b = max_raw(a, b);
    swap_halves32(a, b);
    return max_raw(a, b);
}
__device__ __forceinline__ float xor_sum_g(float v) {
    float a = v, b = v;
    swap_rows16(a, b);
    a = b = a + b;
    swap_halves32(a, b);
    return a + b;
}

// acc + the two 16-bit floats of `w` (one instruction: a dot product with (1, 1))
template <int DT>
__device__ __forceinline__ float add_pair(uint32_t w, float acc) {
    if (DT == DT_F16) {
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, w), __builtin_bit_cast(h2, 0x3c003c00u), acc, false);
    }
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, w), __builtin_bit_cast(b2, 0x3f803f80u), acc, false);
}

// f32 -> cache-type bits, two values at a time
template <int DT>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    if (DT == DT_F16) {
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, h2{(_Float16)a, (_Float16)b});
    }
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, b2{(__bf16)a, (__bf16)b});
}

// Straight into LDS: one instruction moves 64 x 16 bytes from
// per-lane global addresses to 1024 consecutive bytes of LDS at a wave-uniform address; no registers, no LDS stores.
__device__ __forceinline__ void dma16(const uint8_t* src, uint8_t* lds_dst) {
    typedef __attribute__((address_space(3))) void* lds_p;
    typedef const __attribute__((address_space(1))) void* glb_p;
    __builtin_amdgcn_global_load_lds((glb_p)src, (lds_p)lds_dst, 16, 0, 0);
}
// Workgroup barrier for LDS traffic only.  __syncthreads() (and a workgroup fence of any kind) makes the compiler wait
// for every copy into LDS that is in flight, the prefetched blocks included; here the wave waits for its own LDS
// operations, meets the others, and the copies it must have finished are named by the caller (wait_vmem).  The
// barrier instruction and the empty asm statements keep the compiler from moving LDS accesses across.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0); vmcnt and expcnt at their maxima
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
// Waits until at most N of the wave's vector-memory operations are outstanding (gfx9 encoding: vmcnt in bits 3:0 and
// 15:14; the other counters left at their maxima).
template <int N>
__device__ __forceinline__ void wait_vmem() {
    __builtin_amdgcn_s_waitcnt((N & 0xf) | ((N >> 4) << 14) | 0x0f70);
}

}  // namespace
}  // namespace pa
