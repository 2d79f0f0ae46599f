// The Q8_0 prefill tiles: y[M, N] = x[M, K] (f16) . W[N, K]^T, K a multiple of
// 256, operands 16-byte aligned (launched from kquant_prefill.hip).
//
// A workgroup of 4 x 2 waves computes a 32 TM x 128 tile over one part of K;
// wave (kg, wn) multiplies all 32 TM token rows with its own 32 weight rows over
// one half of the part.  The weight operand is the block's bytes v as binary16
// integers, exact, so every product with an activation is exact in f32; a
// block's 32 products per output are two v_mfma_f32_32x32x16_f16 from zero, and
//   y += d C
// in f32 once per block.  (The tiles of q4_0_prefill.hip carry v d as binary16
// hi + lo, four MFMAs per block, and stay for other K and alignments.)
//
// Outputs that are not finite: with a finite scale a block's d C is infinite or
// NaN just where its sum of (v d) x is.  With an infinite one, d C is NaN where C
// is 0, and so is that sum (it has a zero or both signs); else d C is infinite,
// where a zero value or activation, or both signs, make the sum NaN.  So a NaN
// stands, and an infinity does unless one of the row's scales is not finite: then
// those blocks are added up element by element.  (Recomputing every such output
// by its thread took 30 ms where 300 x 4096 x 4096 has NaN activations.)
//
// An interval is 64 k (a block pair) of each half with one barrier, as in
// q4_0_prefill_ring.hip: activations in three slots of swizzled 128-byte rows;
// weights in two slots private to the wave, the five 16-byte chunks that hold
// pair p = 0..3 of each row's 272-byte super-pair.  Both half waves read row r's
// chunks (dword offset p) and lane (r, c) keeps bytes 16 c .. 16 c + 15 of both
// blocks.  Loaded to registers directly, 16 unaligned bytes of 32 rows per
// instruction, the same arithmetic took 145 us instead of 94 at 512 x 4096 x 14
// 336: every lane's address costs the memory pipe a cycle.
//
// Measured on MI355X (weights of three calls rotated), the tiles of
// q4_0_prefill.hip against these: 300 x 4096 x 14 336 88.3 -> 69.0 us, 512 x 4096
// x 14 336 106.7 -> 93.6, 1024 x 14 336 x 4096 214 -> 155, 256 x 14 336 x 4096
// 100 -> 52, 256 x 4096 x 4096 32 -> 22, 48 x 8192 x 28 672 80 -> 75; relative
// error against 64 bits 5.7e-7 -> 1.5e-7 at K = 4096.  Bound by the vector
// pipe: 16 fmas per tile and block beside two MFMAs, and 10 instructions per 8
// weights; counters have 14 to 15 vector instructions per MFMA and MFMAs in 25 to
// 27 % of all SIMD cycles.
#pragma once

#include "kquant_blocks.hpp"
#include "tile_ops.hpp"

#include <type_traits>

namespace mote::kquant {
namespace {

// Whether one of `blocks` block scales from `row` on is not finite.
__device__ inline bool q8_scales_not_finite(const uint8_t* row, uint32_t blocks) {
    bool any = false;
#pragma unroll 8
    for (uint32_t b = 0; b < blocks; ++b)
        any |= (*reinterpret_cast<const uint16_t*>(row + b * 34u) & 0x7C00u) == 0x7C00u;
    return any;
}
// The output that came out as the infinity v: NaN if the sum over a block whose
// scale is not finite is.
__device__ inline float q8_infinite(float v, const uint8_t* row, const uint16_t* xrow, uint32_t blocks) {
    for (uint32_t b = 0; b < blocks; ++b) {
        if (!q8_scales_not_finite(row + b * 34u, 1)) continue;
        float s = 0.0f;
        for (uint32_t e = 0; e < 32; ++e)
            s += half_bits_to_float(xrow[b * 32 + e]) * kq_value<Fmt::Q8>(row + b * 34u, e);
        if (s != s) return s;
    }
    return v;
}

template <int TM, bool SK, typename OutT>
__global__ __launch_bounds__(512) void q8_prefill_kernel(const uint16_t* __restrict__ x, const uint8_t* __restrict__ w,
                                                         OutT* __restrict__ y, float* __restrict__ partial, uint32_t M,
                                                         uint32_t N, uint32_t K, uint32_t m_tiles, uint32_t n_tiles,
                                                         uint32_t part_blocks, uint32_t total, uint32_t per_xcd) {
    constexpr int WN = 4, KG = 2, W = WN * KG;
    constexpr int BM = 32 * TM;
    constexpr int kUnit = BM * 128;          // LDS bytes of one half's activations of an interval
    constexpr int kSlotsX = 3, kSlotsW = 2;
    constexpr int NX = BM / (8 * WN);        // activation loads per wave and interval
    constexpr int NW = 3;                    // weight loads: 32 rows x 5 chunks, and 32 repeats of the last
    constexpr int kWaveW = NW * 1024;
    constexpr int kRingX = kSlotsX * KG * kUnit;
    constexpr uint32_t BB = 272;
    static_assert(W * ((TM + 1) / 2) * 4096 <= kRingX, "the reduction fits the ring");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kRingX + kSlotsW * W * kWaveW];

    const uint32_t logical = (blockIdx.x % 8u) * per_xcd + blockIdx.x / 8u;
    if (logical >= total) return;
    const uint32_t tile_m = logical % m_tiles, rest = logical / m_tiles;
    const uint32_t tile_n = rest % n_tiles, part = rest / n_tiles;
    const uint32_t m0 = tile_m * BM, n0 = tile_n * 128;
    const uint32_t nb = K / kSuper;
    const uint32_t pb0 = part * part_blocks, pb1 = min(pb0 + part_blocks, nb);
    const int lane = static_cast<int>(threadIdx.x) & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int kg = wave / WN, wn = wave % WN;
    const int lr = lane & 31, lc = lane >> 5;
    // this half's super-pairs: [b0, b0 + ns)
    const uint32_t per = (pb1 - pb0 + KG - 1) / KG;
    const uint32_t b0 = min(pb0 + static_cast<uint32_t>(kg) * per, pb1);
    const uint32_t ns = min(per, pb1 - b0);
    const uint32_t last = ns * 4 - 1;  // (no loads where ns is 0)
    const uint32_t row_bytes = nb * BB;

    const Buffer xsrc = buffer_at(reinterpret_cast<const uint8_t*>(x) + (static_cast<size_t>(m0) * K + b0 * kSuper) * 2);
    uint32_t xoff[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
        const uint32_t row = (wn * NX + i) * 8 + (lane >> 3);
        xoff[i] = (min(m0 + row, M - 1) - m0) * (K * 2) + (((lane & 7) ^ ((row >> 1) & 7)) * 16);
    }
    const Buffer wsrc = buffer_at(w + static_cast<size_t>(n0) * row_bytes + b0 * BB);
    uint32_t woff[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        const uint32_t at = min(64u * i + lane, 159u), row = at / 5, c = at % 5;
        woff[i] = (min(n0 + wn * 32 + row, N - 1) - n0) * row_bytes + c * 16;
    }
    uint8_t* const unit = lds + kg * kUnit;
    uint8_t* const own = lds + kRingX + wave * kWaveW;
    auto load_x = [&](uint32_t t, uint32_t slot) {  // interval t (clamped)
        const uint32_t o = min(t, last) * 128u;
#pragma unroll
        for (int i = 0; i < NX; ++i)
            load_lds16(xsrc, xoff[i], o, unit + slot * (KG * kUnit) + (wn * NX + i) * 1024);
    };
    auto load_w = [&](uint32_t t, uint32_t slot) {
        t = min(t, last);
        const uint32_t o = (t >> 2) * BB + (t & 3u) * 64u;  // the chunk pair t % 4 starts in
        uint8_t* const dst = own + slot * (W * kWaveW);
#pragma unroll
        for (int i = 0; i < NW; ++i) load_lds16(wsrc, woff[i], o, dst + i * 1024);
    };

    f32x16 acc[TM], blk[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = blk[i][r] = 0.0f;
    const f32x16 zero = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    f16x8 a[2][TM], b[2];
    uint32_t raw[20], q[2][4];
    float d[2] = {0.0f, 0.0f}, d_before = 0.0f;  // the pair's scales, the pair before's second
    const uint32_t a_row = lr * 128, a_x = (lr >> 1) & 7;
    auto read_x = [&](uint32_t slot, int s, f16x8 (&dst)[TM]) {
        const uint8_t* base = unit + slot * (KG * kUnit) + a_row + (((4 * (s >> 1) + 2 * lc + (s & 1)) ^ a_x) * 16);
#pragma unroll
        for (int i = 0; i < TM; ++i) dst[i] = *reinterpret_cast<const f16x8*>(base + i * 4096);
    };
    auto read_w = [&](uint32_t slot) {
        const uint8_t* base = own + slot * (W * kWaveW) + lr * 80;
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(base + 16 * i);
            raw[4 * i] = v.x; raw[4 * i + 1] = v.y; raw[4 * i + 2] = v.z; raw[4 * i + 3] = v.w;
        }
    };
    // The pair at dword P of the chunks read: this lane's 16 bytes of its two
    // blocks (as v + 128) and both scales.
    auto unpack = [&](auto pc) {
        constexpr int P = decltype(pc)::value;
        auto mine = [&](int low, int high) {  // by value: a select of addresses would move raw to memory
            const uint32_t u = raw[P + low], v = raw[P + high];
            return lc ? v : u;
        };
        uint32_t s[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) s[k] = mine(k, 4 + k);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            q[0][k] = perm(s[k + 1], s[k], 0x05040302u) ^ 0x80808080u;
            q[1][k] = mine(9 + k, 13 + k) ^ 0x80808080u;
        }
        d[0] = half_lo_to_float(raw[P]);
        d[1] = half_hi_to_float(raw[P + 8]);
        asm("" : "+v"(d[0]), "+v"(d[1]));  // kept in f32: mixed-precision fmas need a wait state each
    };
    // Slice s: eight bytes of block s / 2, as binary16 1024 + (v + 128) - 1152.
    auto decode = [&](auto sc, f16x8& dst) {
        constexpr int S = decltype(sc)::value;
        const uint32_t q0 = q[S / 2][2 * (S % 2)], q1 = q[S / 2][2 * (S % 2) + 1], e = 0x64646464u;
        const f16x2 o = both(static_cast<_Float16>(-1152.0f));
        dst = join(as_h2(perm(e, q0, 0x04010400u)) + o, as_h2(perm(e, q0, 0x04030402u)) + o,
                   as_h2(perm(e, q1, 0x04010400u)) + o, as_h2(perm(e, q1, 0x04030402u)) + o);
    };
    auto fold = [&](int i, float by) {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = __builtin_fmaf(by, blk[i][r], acc[i][r]);
    };
    // A block's first slice: the sums of the block before join the result, tile
    // by tile ahead of the tile's product.
    auto multiply_first = [&](float by) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            fold(i, by);
            blk[i] = mfma32(a[0][i], b[0], zero);
        }
    };
    auto multiply = [&]() {
#pragma unroll
        for (int i = 0; i < TM; ++i) blk[i] = mfma32(a[1][i], b[1], blk[i]);
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;

    if (ns > 0) {  // uniform over the wave; a half without work only meets the barriers
        load_x(0, 0);
        order_fence();
        load_w(0, 0);
        order_fence();
        load_x(1, 1);
        order_fence();
        load_w(1, 1);
        order_fence();
        load_x(2, 2);
        order_fence();
        wait_counts<vm_wait(2 * NX + NW)>();
    }
    group_barrier();
    order_fence();
    if (ns > 0) {
        read_w(0);
        read_x(0, 0, a[0]);
        unpack(I0{});
        wait_counts<kLgkmWait>();
        order_fence();
        decode(I0{}, b[0]);
        uint32_t slot = 0, t = 0;
        auto interval = [&](auto pc) {
            constexpr int P = decltype(pc)::value;
            using PN = std::integral_constant<int, (P + 1) & 3>;
            const uint32_t next = slot == kSlotsX - 1 ? 0 : slot + 1;
            load_w(t + 2, P & 1);  // this interval's pairs are in registers
            memory_fence();
            read_x(slot, 1, a[1]);
            multiply_first(d_before);
            decode(I1{}, b[1]);
            order_fence();
            read_x(slot, 2, a[0]);
            multiply();
            decode(I2{}, b[0]);
            order_fence();
            read_x(slot, 3, a[1]);
            // interval t + 1 has landed (at most t + 2's loads are outstanding)
            wait_counts<vm_wait(NX + NW)>();
            memory_fence();
            read_w((P + 1) & 1);
            multiply_first(d[0]);
            decode(I3{}, b[1]);
            order_fence();
            // ... for every wave, and every wave has read interval t
            wait_counts<kLgkmWait>();
            group_barrier();
            order_fence();
            read_x(next, 0, a[0]);
            load_x(t + 3, slot);
            memory_fence();
            multiply();
            d_before = d[1];
            unpack(PN{});
            decode(I0{}, b[0]);
            order_fence();
            slot = next;
            ++t;
        };
        for (uint32_t s = 0; s < ns; ++s) {
            interval(I0{});
            interval(I1{});
            interval(I2{});
            interval(I3{});
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) fold(i, d_before);
    }
    for (uint32_t t = ns * 4; t < per * 4; ++t) group_barrier();
    wait_counts<vm_wait(0)>();
    __syncthreads();

    // The first half keeps row tiles 0 .. H - 1, the second the others; each
    // hands over the rest.
    constexpr int H = (TM + 1) / 2;
    const int kept = kg == 0 ? H : TM - H, tile0 = kg == 0 ? 0 : H;
    float* red = reinterpret_cast<float*>(lds);
    auto place = [&](int wv, int i, int r) { return red + ((wv * H + i) * 4 + r) * 256 + lane * 4; };
    auto give = [&](const f32x16& v, int i) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            *reinterpret_cast<f32x4*>(place(wave, i, r)) = f32x4{v[4 * r], v[4 * r + 1], v[4 * r + 2], v[4 * r + 3]};
    };
    if (kg == 0) {
#pragma unroll
        for (int i = 0; i < TM - H; ++i) give(acc[H + i], i);
    } else {
#pragma unroll
        for (int i = 0; i < H; ++i) {
            give(acc[i], i);
            if (H + i < TM) acc[i] = acc[H + i];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < H; ++i) {
        if (i >= kept) break;  // uniform
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(place(wave ^ WN, i, r));
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[i][4 * r + k] += v[k];
        }
    }
    // Lane (r, c) holds column r of each tile, rows 8 (k / 4) + 4 c + k % 4.
    const uint32_t n = n0 + wn * 32 + lr;
    if (n >= N) return;
    const uint8_t* const wrow = w + (static_cast<size_t>(n) * nb + pb0) * BB;
    const uint32_t blocks = (pb1 - pb0) * 8;
    auto infinite = [](float v) { return (__builtin_bit_cast(uint32_t, v) & 0x7FFFFFFFu) == 0x7F800000u; };
    bool inf = false;
#pragma unroll
    for (int i = 0; i < H; ++i)
#pragma unroll
        for (int k = 0; k < 16; ++k) inf |= i < kept && infinite(acc[i][k]);
    const bool recompute = wave_any(inf) && q8_scales_not_finite(wrow, blocks);
#pragma unroll
    for (int i = 0; i < H; ++i) {
        if (i >= kept) break;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const uint32_t m = m0 + (tile0 + i) * 32 + 8 * (k / 4) + 4 * lc + k % 4;
            if (m >= M) continue;
            float v = acc[i][k];
            if (__builtin_expect(recompute, 0) && infinite(v))
                v = q8_infinite(v, wrow, x + static_cast<size_t>(m) * K + static_cast<size_t>(pb0) * kSuper, blocks);
            if constexpr (SK)
                partial[(static_cast<size_t>(part) * M + m) * N + n] = v;
            else
                y[static_cast<size_t>(m) * N + n] = to_out<OutT>(v);
        }
    }
}

}  // namespace
}  // namespace mote::kquant
