// K-quant super-blocks as the kernels see them: geometry, the Q4_K scale
// packing, unaligned 16-byte reads, and GGML's per-element values, from which
// a row whose folded sum is not finite is recomputed.  Layouts: kquant.hip.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"

namespace mote::kquant {

// (Q8: eight consecutive Q8_0 blocks, 256 elements in 272 bytes; many-token
// linear only.)
enum class Fmt { Q4K, Q6K, Q8 };

namespace {

constexpr uint32_t kSuper = 256;

template <Fmt F>
constexpr uint32_t block_bytes() {
    return F == Fmt::Q4K ? 144u : F == Fmt::Q6K ? 210u : 272u;
}

__device__ __forceinline__ float half_bits_to_float(uint32_t bits) {
    return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(bits)));
}

// Sub-block j's 6-bit scale and min from the three dwords holding the 12
// scale bytes (s0 = s[0..3], s1 = s[4..7], s2 = s[8..11]).
__device__ __forceinline__ void q4k_scale_min(uint32_t s0, uint32_t s1, uint32_t s2, uint32_t j, uint32_t& sc,
                                              uint32_t& m) {
    const uint32_t sh = 8u * (j & 3u);
    const uint32_t a = __builtin_amdgcn_ubfe(s0, sh, 8), b = __builtin_amdgcn_ubfe(s1, sh, 8);
    if (j < 4) {
        sc = a & 63u;
        m = b & 63u;
    } else {
        const uint32_t c = __builtin_amdgcn_ubfe(s2, sh, 8);
        sc = (c & 15u) | ((a >> 6) << 4);
        m = (c >> 4) | ((b >> 6) << 4);
    }
}

// 16 bytes at a 2-byte-aligned address, read as five dwords from the dword
// boundary at or below it; the caller guarantees the 20 bytes from there lie
// inside the object.
__device__ __forceinline__ u32x4 load16_a2(const uint8_t* p) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(p);
    const uint32_t* q = reinterpret_cast<const uint32_t*>(a & ~uintptr_t{3});
    const uint32_t sh = static_cast<uint32_t>(a & 3u);  // 0 or 2
    const u32x4_a4 v = *reinterpret_cast<const u32x4_a4*>(q);
    const uint32_t e = q[4];
    u32x4 r;
    r.x = __builtin_amdgcn_alignbyte(v.y, v.x, sh);
    r.y = __builtin_amdgcn_alignbyte(v.z, v.y, sh);
    r.z = __builtin_amdgcn_alignbyte(v.w, v.z, sh);
    r.w = __builtin_amdgcn_alignbyte(e, v.w, sh);
    return r;
}

// ---------------------------------------------------------------------------
// Rows whose sum is not finite.  The linears below fold a sub-block's scale
// and min into sums over its elements (d sc sum x q - dmin m sum x); GGML's
// definition, which the oracle follows, rounds every element's value first
// (d1 = d sc, m1 = dmin m, then d1 q - m1 for Q4_K; (d sc)(q - 32) for
// Q6_K) and sums x times that.  With finite scales and activations neither
// form can overflow, so they agree to rounding; an infinite or NaN scale (or
// a non-finite activation) makes the folded sum not finite, and then it can
// put +-inf where the per-element values give NaN (inf * 0 for q = 0 or
// sc = 0, products of both signs).  (The few-token Q4_K tiles get there with
// finite activations whose sum over a sub-block passes binary16's range, too.)
// A wave whose reduced sum is not finite (a
// wave-uniform test) recomputes its share of the row element by element, so
// the NaN and infinities land where the definition puts them.
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool not_finite(float v) {
    return (__builtin_bit_cast(uint32_t, v) & 0x7F800000u) == 0x7F800000u;
}

// GGML's value of element e (0..255) of the super-block at `blk` (global
// memory), with the oracle's f32 rounding points.
template <Fmt F>
__device__ inline float kq_value(const uint8_t* blk, uint32_t e) {
    if constexpr (F == Fmt::Q4K) {
        const uint32_t p = e >> 6, h = (e >> 5) & 1u, l = e & 31u, j = 2 * p + h;
        const uint8_t* sb = blk + 4;
        uint32_t sc, m;
        if (j < 4) {
            sc = sb[j] & 63u;
            m = sb[j + 4] & 63u;
        } else {
            sc = (sb[j + 4] & 15u) | ((sb[j - 4] >> 6) << 4);
            m = (sb[j + 4] >> 4) | ((sb[j] >> 6) << 4);
        }
        const float d1 = half_bits_to_float(blk[0] | (blk[1] << 8)) * static_cast<float>(sc);
        const float m1 = half_bits_to_float(blk[2] | (blk[3] << 8)) * static_cast<float>(m);
        const uint32_t byte = blk[16 + 32 * p + l];
        const float prod = d1 * static_cast<float>(h ? byte >> 4 : byte & 15u);
        return prod - m1;
    } else if constexpr (F == Fmt::Q8) {
        const uint8_t* b = blk + 34 * (e >> 5);
        return half_bits_to_float(b[0] | (b[1] << 8)) * static_cast<float>(static_cast<int8_t>(b[2 + (e & 31u)]));
    } else {
        const uint32_t g = e >> 7, c = (e >> 5) & 3u, l = e & 31u;
        const uint32_t low = blk[64 * g + 32 * (c & 1u) + l] >> (4 * (c >> 1)) & 15u;
        const uint32_t high = (blk[128 + 32 * g + l] >> (2 * c)) & 3u;
        const float ds = half_bits_to_float(blk[208] | (blk[209] << 8)) *
                         static_cast<float>(static_cast<int8_t>(blk[192 + e / 16]));
        return ds * static_cast<float>(static_cast<int>(low | (high << 4)) - 32);
    }
}

// sum over the row of x[k] w[k] with GGML's per-element values, one thread.
template <Fmt F>
__device__ inline float kq_exact_thread(const uint8_t* row, const uint16_t* xrow, uint32_t nb) {
    float acc = 0.0f;
    for (uint32_t k = 0; k < nb * kSuper; ++k)
        acc += half_bits_to_float(xrow[k]) *
               kq_value<F>(row + static_cast<size_t>(k / kSuper) * block_bytes<F>(), k % kSuper);
    return acc;
}

}  // namespace

int device_cus();

// The linear over many tokens on the matrix cores (kquant_prefill.hip):
// whether it takes the call, and the call (F16: binary16 result).  On a stream
// without prompt scratch (q4_0.hpp) it runs over all of K at once, except for up
// to 64 tokens: hipErrorNotSupported, with nothing queued.
bool prefill_supported(Fmt f, const void* x, const void* w, uint32_t M, uint32_t N, uint32_t K);
hipError_t launch_prefill(Fmt f, bool f16_out, const void* x, const void* w, void* y, uint32_t M, uint32_t N,
                          uint32_t K, hipStream_t stream);

}  // namespace mote::kquant
