// What the direct-to-LDS prefill tiles share: counted waits, the 32 x 32 x 16
// MFMA, loads to LDS, packed binary16 helpers, the sum over K parts.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"

namespace mote {
namespace {

// s_waitcnt immediates: until at most n vector memory loads are outstanding
// (they count in issue order); lgkmcnt(0) alone.  ANDed: both.
constexpr int vm_wait(int n) { return (n & 0xF) | ((n >> 4) << 14) | 0x0F70; }
constexpr int kLgkmWait = 0xC07F;

// The builtins behind plain functions (usable from generic lambdas).  Loads to
// LDS by buffer address where loads to registers are in flight beside them:
// those by global address make the compiler wait for every load (vmcnt(0))
// before it uses one's result.
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __amdgpu_buffer_rsrc_t Buffer;
__device__ __forceinline__ Buffer buffer_at(const void* base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, 0xFFFFFFFFu, 0x00020000);
}
__device__ __forceinline__ void load_lds16(Buffer src, uint32_t lane_offset, uint32_t offset, uint8_t* dst) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (lds_ptr_t)dst, 16, lane_offset, offset, 0, 0);
}
__device__ __forceinline__ void load_lds16(const uint8_t* src, uint8_t* dst) {
    __builtin_amdgcn_global_load_lds(src, (lds_ptr_t)dst, 16, 0, 0);
}
template <int I>
__device__ __forceinline__ void wait_counts() { __builtin_amdgcn_s_waitcnt(I); }
__device__ __forceinline__ void order_fence() { __builtin_amdgcn_sched_barrier(0); }
// Keeps memory operations on their side of this point, in the compiler's
// intermediate code and in its schedule: counted waits rely on the
// order in which the loads are issued.
__device__ __forceinline__ void issue_fence() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void group_barrier() { __builtin_amdgcn_s_barrier(); }
__device__ __forceinline__ f32x16 mfma32(const f16x8& a, const f16x8& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) {
    return __builtin_amdgcn_perm(hi, lo, sel);
}
__device__ __forceinline__ f16x2 both(f16x2 v, bool high) {
    const uint32_t b = __builtin_bit_cast(uint32_t, v);
    return as_h2(perm(b, b, high ? 0x03020302u : 0x01000100u));
}
__device__ __forceinline__ f16x2 both(_Float16 v) { return f16x2{v, v}; }
__device__ __forceinline__ f16x8 join(f16x2 a, f16x2 b, f16x2 c, f16x2 d) {
    return f16x8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}


// y[i] = the sum of the K parts' planes at i, in part order, converted.
template <typename OutT>
__global__ __launch_bounds__(256) void parts_reduce_kernel(const float* __restrict__ partial, uint32_t parts,
                                                              uint64_t count, OutT* __restrict__ y) {
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= count) return;
    float v = partial[i];
    for (uint32_t k = 1; k < parts; ++k) v += partial[k * count + i];
    y[i] = to_out<OutT>(v);
}

}  // namespace
}  // namespace mote
