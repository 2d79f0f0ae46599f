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
// Keeps memory operations on their side of this point, in the compiler's
// intermediate code and in its schedule: counted waits rely on the
// order in which the loads are issued, LDS reads on staying behind the wait and
// the barrier that their data needs.
__device__ __forceinline__ void memory_fence() { asm volatile("" ::: "memory"); }
// ... and everything else on its side in the schedule.
__device__ __forceinline__ void order_fence() {
    memory_fence();
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void group_barrier() { __builtin_amdgcn_s_barrier(); }
__device__ __forceinline__ f32x16 mfma32(const f16x8& a, const f16x8& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ f32x16 mfma32(const bf16x8& a, const bf16x8& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
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


// y[i] = the sum of the K parts' planes at i, in part order, converted; four
// consecutive outputs per thread (16-byte loads and stores at the planes' 4- and
// the output's element alignment; against one per thread, whole calls: 256 x 14
// 336 x 4096 Q4_0 43.7 -> 43.0 us, Q6_K 62.9 -> 62.0, Q8_0 48.5 -> 47.8).
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef _Float16 f16x4_a2 __attribute__((ext_vector_type(4), aligned(2)));

template <typename OutT>
__global__ __launch_bounds__(256) void parts_reduce_kernel(const float* __restrict__ partial, uint32_t parts,
                                                           uint64_t count, OutT* __restrict__ y) {
    const uint64_t i = (static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
    if (i + 4 <= count) {
        f32x4 v = *reinterpret_cast<const f32x4_a4*>(partial + i);
        for (uint32_t k = 1; k < parts; ++k) v += *reinterpret_cast<const f32x4_a4*>(partial + k * count + i);
        if constexpr (sizeof(OutT) == 4)
            *reinterpret_cast<f32x4_a4*>(y + i) = v;
        else
            *reinterpret_cast<f16x4_a2*>(y + i) =
                f16x4_a2{to_out<OutT>(v.x), to_out<OutT>(v.y), to_out<OutT>(v.z), to_out<OutT>(v.w)};
        return;
    }
    for (uint64_t e = i; e < count; ++e) {
        float v = partial[e];
        for (uint32_t k = 1; k < parts; ++k) v += partial[k * count + e];
        y[e] = to_out<OutT>(v);
    }
}

// Its grid: 1024 outputs per workgroup.
inline uint32_t parts_reduce_grid(uint64_t count) { return static_cast<uint32_t>((count + 1023) / 1024); }

}  // namespace
}  // namespace mote
