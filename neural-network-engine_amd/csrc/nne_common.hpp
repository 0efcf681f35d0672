// Shared device helpers of the attention kernels; the launch-parameter
// structs and layout conventions are in nne_params.hpp.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "nne_params.hpp"

namespace nne {

typedef float floatx16 __attribute__((ext_vector_type(16)));
// Native 4-float vector for register tiles and 16-byte loads/stores.  (HIP's
// float4 is a struct whose copies lower to memcpy through private memory,
// which can keep register arrays of it out of registers.)
typedef float vf4 __attribute__((ext_vector_type(4)));

// Operand of a bf16 MFMA: 8 values of one lane.
typedef short short8 __attribute__((ext_vector_type(8)));
typedef float vf2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegInf = -__builtin_huge_valf();

// ---- f32 products on the bf16 matrix cores -----------------------------------
// An f32 value is the exact sum of three bf16 values (8 significant bits and a
// sign each, rounded to nearest: 24 bits in all), and the product of two of
// them is nine bf16 products.  The six largest are computed,
//   xy = hh + (hm + mh) + (mm + hl + lh) + O(2^-25 |xy|),
// each product exact and every sum in f32, as on the f32 MFMAs; with h, m and
// l the high, middle and low parts.  gfx950's bf16 MFMAs run at 16x the rate
// of its f32 ones, so six of them take 3/8 of the time (measured on registers:
// 1777 / 6 = 296 against 146 TFLOP/s), and their sums are rounded less often:
// the error of a 128-term dot product of N(0, 1) values against 64 bits is
// 0.7e-7 to 1.6e-7 (two accumulators, one) where the f32 MFMAs give 2.0e-7.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(vf2{a, b}, bf16x2));
}
// The three parts of a (low 16 bits) and b (high 16 bits).
__device__ __forceinline__ void split3(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
    h = pack_bf16(a, b);
    a -= __uint_as_float(h << 16);
    b -= __uint_as_float(h & 0xffff0000u);
    m = pack_bf16(a, b);
    a -= __uint_as_float(m << 16);
    b -= __uint_as_float(m & 0xffff0000u);
    l = pack_bf16(a, b);
}
__device__ __forceinline__ floatx16 mfma_bf16(short8 a, short8 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// The conversions and the MFMAs keep bf16's subnormals, so the parts hold a value
// down to 2^-133, whole from 2^-110 up.  Softmax weights come as small as 2^-126
// and are split 2^16 times their size (a weight of 2^-124 on a V beyond 2^100
// times the others' is a result like any other: without it 3e-4 of error there),
// and so is V, whose parts are then whole at any size (subnormals are multiples
// of 2^-133; unscaled, a V of 1e-42 gave zeros).
// Where the parts do not hold a value: an infinity, a NaN or a magnitude that
// rounds or grows to infinity leaves NaN parts, and every result it enters is not
// finite.  A tiny query that meets a huge key, or a huge query that meets a tiny
// key, does not show there, so queries have a range of their own.
// (range_code: 0 for zero, ascending with the magnitude from 2^-110 on, above
// every such code for smaller magnitudes.)
__device__ __forceinline__ uint32_t range_code(float x) {
    const uint32_t a = __float_as_uint(x) & 0x7fffffffu;
    return a == 0 ? 0 : a - __float_as_uint(0x1p-110f);
}
constexpr float kPartUp = 0x1p16f, kPartDown = 0x1p-32f;   // of a weight or value, of their product
constexpr uint32_t kQueryCodes = 0x6c800000u - 0x08800000u;    // codes of queries up to 2^90

// Brings [B0, E0) and [B1, E1) of the kernel argument block into the scalar
// cache: one load per 64-byte line, all issued before a single wait.  The
// arguments read later then hit there instead of each first use paying a
// memory round trip in a dependent chain (about 1 us apiece at a launch).
template <int B0, int E0, int B1, int E1>
__device__ __forceinline__ void warm_kernargs() {
    typedef const __attribute__((address_space(4))) int kernarg_int;
    kernarg_int* kp = (kernarg_int*)__builtin_amdgcn_kernarg_segment_ptr();
    constexpr int N0 = (E0 - B0 + 63) / 64, N1 = (E1 - B1 + 63) / 64;
    int v[N0 + N1];
#pragma unroll
    for (int i = 0; i < N0; ++i) v[i] = kp[(B0 + 64 * i) / 4];
#pragma unroll
    for (int i = 0; i < N1; ++i) v[N0 + i] = kp[(B1 + 64 * i) / 4];
#pragma unroll
    for (int i = 0; i < N0 + N1; ++i) asm volatile("" ::"s"(v[i]));
}
template <int B0, int E0>
__device__ __forceinline__ void warm_kernargs() {
    warm_kernargs<B0, E0, E0, E0>();
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Partial records cross workgroups without a fence: they are written with
// agent-scope relaxed atomic stores (global_store sc1, written through to the
// device coherence point) and read with agent-scope relaxed atomic loads
// (global_load sc1, never served from a stale per-XCD L2 line).  A writer waits
// for its stores (vmcnt(0)) before its arrival is counted, and a reader loads
// only after the count says every writer has arrived.  An agent-scope
// release/acquire pair would also write back and invalidate the whole L2 of
// each XCD, which costs tens of microseconds per launch.
__device__ __forceinline__ void store_coherent(float* p, float x) {
    __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_coherent(const float* p) {
    return __hip_atomic_load(const_cast<float*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// 16-byte form of load_coherent: a buffer load with the same sc1 policy
// (buffer_load_dwordx4 ... sc1) from a range of `bytes` bytes at `base`
// (offsets past the range read as zero).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t coherent_range(const float* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, bytes, 0x00020000);
}
__device__ __forceinline__ vf4 load_coherent4(__amdgpu_buffer_rsrc_t range, uint32_t byte_offset) {
    return __builtin_bit_cast(vf4, __builtin_amdgcn_raw_buffer_load_b128(range, byte_offset, 0, 16));
}
__device__ __forceinline__ float2 load_coherent2(__amdgpu_buffer_rsrc_t range, uint32_t byte_offset) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b64(range, byte_offset, 0, 16);
    return float2{__uint_as_float(v[0]), __uint_as_float(v[1])};
}
__device__ __forceinline__ void wait_stores_performed() {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0), expcnt/lgkmcnt unconstrained
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}


// Swaps lanes 32..63 of `a` with lanes 0..31 of `b` (gfx950 v_permlane32_swap).
// Called with a == b == x, element 0 of the result holds x from lanes 0..31 in
// both halves and element 1 holds x from lanes 32..63 in both halves, so
// combining the two elements reduces over the lane pair (l, l ^ 32).
__device__ __forceinline__ float pair_max(float x) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

__device__ __forceinline__ float pair_sum(float x) {
    auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

}  // namespace nne
