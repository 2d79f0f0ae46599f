// Q4_0 prefill tiles whose operands come through direct-to-LDS rings, with the
// workgroup's waves split over K: the linear and the fused gate/up of
// q4_0_prefill.hip for K a multiple of 256 and 16-byte-aligned operands.
//
// A workgroup of WN x 2 waves computes a 32 TM x 64 WN tile (gate/up: 32 WN
// columns of each).  Wave (kg, wn) multiplies all 32 TM token rows with its own
// 64 weight rows (tile j: rows 32 j ..; gate/up: 32 gate and the same 32 up
// rows) over one half of K: TM x 2 tiles of v_mfma_f32_32x32x16_f16.  So every
// weight is decoded by one wave, once per 32 TM tokens, two waves share each
// SIMD (WN = 4; the 128-column tiles, WN = 2, have one wave per SIMD and 120 KB of
// LDS, so they pay 2.2 us per super-pair where the 256-column ones pay 3.6), and
// the two halves' accumulators meet in LDS at the end.
//
// An interval is 64 k (a block pair) of each half, with one barrier:
//  * activations: 16-byte chunks in their natural order, three slots (two
//    intervals in flight), 128-byte rows, chunks XOR-swizzled by half the row
//    so the 16 rows an operand read covers per cycle fall on the 64 banks once;
//  * weights: the three 16-byte chunks that hold pair p = 0..3 of each row's
//    144-byte super-pair (256 k), two slots, private to the wave.  Lane l reads
//    row l's pair (dword offset p: the same in every lane, a constant of the
//    unrolled loop), and v_permlane32_swap hands block 0 of rows 32.. to the
//    lower and block 1 of rows 0..31 to the upper lanes: lane (r, c) then holds
//    block c of row r of both tiles, and its slice s of four is 8 consecutive
//    elements, low (s < 2) or high nibbles of 8 bytes, the same 8 that the
//    activation operand reads as one chunk.
// The barrier stands before an interval's last slice, whose MFMAs cover the
// next interval's first reads; its weights are read one slice earlier.
//
// Bound by the instruction stream, and the clock falls as it gets denser: counters
// have MFMAs in 42 % of all SIMD cycles at 512 x 4096 x 14 336 (224 workgroups on 256
// CUs) and 46 % in the 1024-token gate/up, and six vector instructions per MFMA.
// Measured on MI355X (weights of three
// calls rotated), the staging-wave body of q4_0_prefill.hip against this one:
// 512 x 4096 x 14 336 66.2 -> 62.7 us, 2048 x 4096 x 4096 73.3 -> 69.7 (128 x
// 256 tiles), 256 x 4096 x 14 336 40.9 -> 38.5, 1024 x 14 336 x 4096 143.7 ->
// 128.1, 400 x 14 336 x 5120 117 -> 98 (128 x 128).  64-row tiles decode each
// weight for half as many MFMAs and measured level or slower than the staging
// waves (128 x 4096 x 14 336 25.1 against 24.8, 64 x 8192 x 28 672 60.9 against
// 53.9; gate/up the same), so they keep those.
#include "common.hpp"
#include "kquant_blocks.hpp"
#include "q4_0.hpp"
#include "tile_ops.hpp"

#include <cmath>
#include <type_traits>

namespace mote::q4_0 {
namespace {

constexpr int kGroups = 2;       // halves of K
constexpr int kSlotsX = 3, kSlotsW = 2;
constexpr int kLoadsW = 3;       // weight loads per wave and interval: 64 rows x 3 chunks
constexpr int kWaveW = 64 * 48;  // their LDS bytes

// x with its upper 32 lanes' values replaced by y's lower ones, and y with its
// lower ones replaced by x's upper ones.
__device__ __forceinline__ u32x2 swap_halves(uint32_t x, uint32_t y) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    return u32x2{r[0], r[1]};
}
// (q - 8) d of the low or high nibbles of the eight bytes q0, q1, in byte
// order: as dequant8 (common.hpp), exact q - 8 from binary16 1024 + q or 64 +
// q, one rounding of the product.
template <bool HIGH>
__device__ __forceinline__ f16x8 dequant8_run(uint32_t q0, uint32_t q1, f16x2 d) {
    constexpr uint32_t mask = HIGH ? 0xF0F0F0F0u : 0x0F0F0F0Fu, e = HIGH ? 0x54545454u : 0x64646464u;
    constexpr float b = HIGH ? -72.0f : -1032.0f;
    const f16x2 bias = {static_cast<_Float16>(b), static_cast<_Float16>(b)};
    const uint32_t t0 = q0 & mask, t1 = q1 & mask;
    const f16x2 v0 = (as_h2(perm(e, t0, 0x04010400u)) + bias) * d;
    const f16x2 v1 = (as_h2(perm(e, t0, 0x04030402u)) + bias) * d;
    const f16x2 v2 = (as_h2(perm(e, t1, 0x04010400u)) + bias) * d;
    const f16x2 v3 = (as_h2(perm(e, t1, 0x04030402u)) + bias) * d;
    return f16x8{v0.x, v0.y, v1.x, v1.y, v2.x, v2.y, v3.x, v3.y};
}

template <int TM, int WN, bool GATE_UP, bool SK, typename OutT>
__global__ __launch_bounds__(64 * WN * kGroups) void prefill_ring_kernel(
    const uint16_t* __restrict__ x, const uint8_t* __restrict__ wg, const uint8_t* __restrict__ wu,
    OutT* __restrict__ y, float* __restrict__ partial, uint32_t M, uint32_t N, uint32_t K, uint32_t m_tiles,
    uint32_t n_tiles, uint32_t part_pairs, uint32_t total, uint32_t per_xcd) {
    constexpr int W = WN * kGroups;
    constexpr int BM = 32 * TM;
    constexpr uint32_t BN = (GATE_UP ? 32 : 64) * WN;  // output columns
    constexpr int kUnit = BM * 128;                    // LDS bytes of one half's activations of an interval
    constexpr int NX = BM / (8 * WN);                  // activation loads per wave and interval
    constexpr int kRingX = kSlotsX * kGroups * kUnit;
    static_assert(TM % 2 == 0 && kRingX + kSlotsW * W * kWaveW <= 160 * 1024, "LDS");
    static_assert(W * (TM / 2) * 2 * 4096 <= kRingX + kSlotsW * W * kWaveW, "the reduction fits the rings");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kRingX + kSlotsW * W * kWaveW];

    const uint32_t logical = (blockIdx.x % 8u) * per_xcd + blockIdx.x / 8u;
    if (logical >= total) return;
    const uint32_t tile_m = logical % m_tiles, rest = logical / m_tiles;
    const uint32_t tile_n = rest % n_tiles, part = rest / n_tiles;
    const uint32_t m0 = tile_m * BM, n0 = tile_n * BN;
    const int lane = static_cast<int>(threadIdx.x) & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int kg = wave / WN, wn = wave % WN;
    const int lr = lane & 31, lc = lane >> 5;
    const uint32_t nsuper = K >> 8;
    const uint32_t row_bytes = nsuper * 144u;
    // this half of the part's super-pairs: [s0, s0 + ns)
    const uint32_t p0 = part * part_pairs, p1 = min(p0 + part_pairs, nsuper);
    const uint32_t per = (p1 - p0 + kGroups - 1) / kGroups;
    const uint32_t s0 = min(p0 + static_cast<uint32_t>(kg) * per, p1);
    const uint32_t ns = min(per, p1 - s0);
    const uint32_t last = ns * 4 - 1;  // (no loads where ns is 0)

    const Buffer xsrc = buffer_at(reinterpret_cast<const uint8_t*>(x) + (static_cast<size_t>(m0) * K + s0 * 256u) * 2);
    uint32_t xoff[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
        const uint32_t row = (wn * NX + i) * 8 + (lane >> 3);
        xoff[i] = (min(m0 + row, M - 1) - m0) * (K * 2) + (((lane & 7) ^ ((row >> 1) & 7)) * 16);
    }
    // Weight load i, lane l: chunk (64 i + l) % 3 of the wave's row (64 i + l) / 3
    // (gate/up: rows 0..31 gate, 32..63 up; from two matrices, by address).
    const Buffer wsrc = buffer_at(wg + static_cast<size_t>(n0) * row_bytes + s0 * 144u);
    uint32_t woff[kLoadsW];
    const uint8_t* wptr[kLoadsW];
#pragma unroll
    for (int i = 0; i < kLoadsW; ++i) {
        const uint32_t at = 64u * i + lane, row = at / 3, c = at % 3;
        if constexpr (GATE_UP)
            wptr[i] = (row < 32 ? wg : wu) + static_cast<size_t>(min(n0 + wn * 32 + (row & 31), N - 1)) * row_bytes +
                      s0 * 144u + c * 16;
        else
            woff[i] = (min(n0 + wn * 64 + row, N - 1) - n0) * row_bytes + c * 16;
    }
    uint8_t* const unit = lds + kg * kUnit;
    uint8_t* const own = lds + kRingX + wave * kWaveW;
    auto load_x = [&](uint32_t t, uint32_t slot) {  // interval t (clamped)
        const uint32_t o = min(t, last) * 128u;
#pragma unroll
        for (int i = 0; i < NX; ++i)
            load_lds16(xsrc, xoff[i], o, unit + slot * (kGroups * kUnit) + (wn * NX + i) * 1024);
    };
    auto load_w = [&](uint32_t t, uint32_t slot) {
        t = min(t, last);
        const uint32_t o = (t >> 2) * 144u + (t & 3u) * 32u;  // the chunk pair t % 4 starts in
#pragma unroll
        for (int i = 0; i < kLoadsW; ++i) {
            uint8_t* const dst = own + slot * (W * kWaveW) + i * 1024;
            if constexpr (GATE_UP)
                load_lds16(wptr[i] + o, dst);
            else
                load_lds16(wsrc, woff[i], o, dst);
        }
    };

    f32x16 acc[TM][2];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    f16x8 a[2][TM], b[2][2];
    uint32_t raw[12], q[2][4];
    f16x2 d[2];
    bool big = false, scaled = false;  // wave-uniform
    const uint32_t a_row = lr * 128, a_x = (lr >> 1) & 7;
    auto read_x = [&](uint32_t slot, int s, f16x8 (&dst)[TM]) {
        const uint8_t* base = unit + slot * (kGroups * kUnit) + a_row + (((4 * lc + s) ^ a_x) * 16);
#pragma unroll
        for (int i = 0; i < TM; ++i) dst[i] = *reinterpret_cast<const f16x8*>(base + i * 4096);
    };
    auto read_w = [&](uint32_t slot) {
        const uint8_t* base = own + slot * (W * kWaveW) + lane * 48;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(base + 16 * i);
            raw[4 * i] = v.x; raw[4 * i + 1] = v.y; raw[4 * i + 2] = v.z; raw[4 * i + 3] = v.w;
        }
    };
    // The pair at dword P of the chunks read: nibble dwords and scales of this
    // lane's block of both tiles.  Scales past binary16 range (common.hpp): the
    // interval runs with every scale of the wave and the accumulators times 2^-4.
    auto unpack = [&](auto pc) {
        constexpr int P = decltype(pc)::value;
        const uint32_t* p = raw + P;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const u32x2 v = swap_halves(perm(p[k + 1], p[k], 0x05040302u), p[5 + k]);
            q[0][k] = v.x;
            q[1][k] = v.y;
        }
        const u32x2 v = swap_halves(p[0], p[4] >> 16);
        const uint32_t d0 = perm(v.x, v.x, 0x01000100u), d1 = perm(v.y, v.y, 0x01000100u);
        d[0] = as_h2(d0);
        d[1] = as_h2(d1);
        big = wave_any(big_scales<kQ4BigScale>(d0) || big_scales<kQ4BigScale>(d1));
        if (__builtin_expect(big, 0)) {
            const f16x2 down = {static_cast<_Float16>(kQ4BigDown), static_cast<_Float16>(kQ4BigDown)};
            d[0] *= down;
            d[1] *= down;
        }
    };
    auto rescale = [&](float f) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] *= f;
    };
    auto decode = [&](auto sc, f16x8 (&dst)[2]) {
        constexpr int S = decltype(sc)::value;
#pragma unroll
        for (int j = 0; j < 2; ++j) dst[j] = dequant8_run<(S > 1)>(q[j][2 * (S & 1)], q[j][2 * (S & 1) + 1], d[j]);
    };
    auto multiply = [&](int cur) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = mfma32(a[cur][i], b[cur][j], acc[i][j]);
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
        wait_counts<vm_wait(2 * NX + kLoadsW)>();
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
            if (__builtin_expect(big != scaled, 0)) {
                scaled = big;
                rescale(big ? kQ4BigDown : 1.0f / kQ4BigDown);
            }
            load_w(t + 2, P & 1);  // this interval's pairs are in registers
            memory_fence();
            read_x(slot, 1, a[1]);
            multiply(0);
            decode(I1{}, b[1]);
            order_fence();
            read_x(slot, 2, a[0]);
            multiply(1);
            decode(I2{}, b[0]);
            order_fence();
            read_x(slot, 3, a[1]);
            // interval t + 1 has landed (at most t + 2's loads are outstanding)
            wait_counts<vm_wait(NX + kLoadsW)>();
            memory_fence();
            read_w((P + 1) & 1);
            multiply(0);
            decode(I3{}, b[1]);
            order_fence();
            // ... for every wave, and every wave has read interval t
            wait_counts<kLgkmWait>();
            group_barrier();
            order_fence();
            read_x(next, 0, a[0]);
            load_x(t + 3, slot);
            memory_fence();
            multiply(1);
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
        if (__builtin_expect(scaled, 0)) rescale(1.0f / kQ4BigDown);
    }
    for (uint32_t t = ns * 4; t < per * 4; ++t) group_barrier();
    wait_counts<vm_wait(0)>();
    __syncthreads();

    // Each half keeps TM / 2 row tiles and hands the others over.
    constexpr int H = TM / 2;
    float* red = reinterpret_cast<float*>(lds);
    auto place = [&](int wv, int i, int j, int r) { return red + (((wv * H + i) * 2 + j) * 4 + r) * 256 + lane * 4; };
    auto give = [&](const f32x16& v, int i, int j) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            *reinterpret_cast<f32x4*>(place(wave, i, j, r)) = f32x4{v[4 * r], v[4 * r + 1], v[4 * r + 2], v[4 * r + 3]};
    };
    if (kg == 0) {
#pragma unroll
        for (int i = 0; i < H; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) give(acc[H + i][j], i, j);
    } else {
#pragma unroll
        for (int i = 0; i < H; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                give(acc[i][j], i, j);
                acc[i][j] = acc[H + i][j];
            }
    }
    __syncthreads();
    const int other = wave ^ WN;
#pragma unroll
    for (int i = 0; i < H; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(place(other, i, j, r));
#pragma unroll
                for (int k = 0; k < 4; ++k) acc[i][j][4 * r + k] += v[k];
            }
    // Lane (r, c) holds column r of each tile, rows 8 (k / 4) + 4 c + k % 4.
#pragma unroll
    for (int j = 0; j < (GATE_UP ? 1 : 2); ++j) {
        const uint32_t n = GATE_UP ? n0 + wn * 32 + lr : n0 + wn * 64 + j * 32 + lr;
        if (n >= N) continue;
#pragma unroll
        for (int i = 0; i < H; ++i)
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const uint32_t m = m0 + (kg * H + i) * 32 + 8 * (k / 4) + 4 * lc + k % 4;
                float v = acc[i][j][k];
                if constexpr (GATE_UP) v = silu(v) * acc[i][1][k];
                if (m >= M) continue;
                if constexpr (SK)  // this K part's plane of the partial sums
                    partial[(static_cast<size_t>(part) * M + m) * N + n] = v;
                else
                    y[static_cast<size_t>(m) * N + n] = to_out<OutT>(v);
            }
    }
}

// parts > 1 (linear): K parts in planes of the stream's prompt scratch, added by
// a second kernel.  hipErrorNotSupported, with nothing queued, where the stream
// has none (acquire_prompt_scratch).
template <int TM, int WN, bool GATE_UP>
hipError_t launch_ring(const Problem& p, uint32_t parts) {
    constexpr uint32_t BM = 32 * TM, BN = (GATE_UP ? 32 : 64) * WN;
    const uint32_t m_tiles = (p.M + BM - 1) / BM;
    const uint32_t n_tiles = (p.N + BN - 1) / BN;
    const uint32_t nsuper = p.K / 256u;
    const uint32_t part_pairs = (nsuper + parts - 1) / parts;
    parts = (nsuper + part_pairs - 1) / part_pairs;
    const uint64_t total64 = static_cast<uint64_t>(m_tiles) * n_tiles * parts;
    if (total64 > 0x7ffffff0ull) return hipErrorInvalidConfiguration;
    const uint32_t total = static_cast<uint32_t>(total64);
    const uint32_t per_xcd = (total + 7u) / 8u;
    const dim3 grid(per_xcd * 8u), block(64 * WN * kGroups);
    const auto* x = static_cast<const uint16_t*>(p.x);
    const auto* wg = static_cast<const uint8_t*>(p.w);
    const auto* wu = static_cast<const uint8_t*>(p.w_up);
    if constexpr (!GATE_UP) {
        if (parts > 1) {
            const uint64_t count = static_cast<uint64_t>(p.M) * p.N;
            ScratchPool::Lease lease;  // holds the scratch until both kernels are queued
            const hipError_t a = acquire_prompt_scratch(p.stream, count * parts * sizeof(float), &lease);
            if (a != hipSuccess) return a;
            auto* const planes = static_cast<float*>(lease.ptr());
            hipLaunchKernelGGL((prefill_ring_kernel<TM, WN, false, true, float>), grid, block, 0, p.stream, x, wg, wu,
                               static_cast<float*>(nullptr), planes, p.M, p.N, p.K, m_tiles, n_tiles, part_pairs, total,
                               per_xcd);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
            const dim3 rgrid(parts_reduce_grid(count)), rblock(256);
            if (p.out == OutType::F32)
                hipLaunchKernelGGL((parts_reduce_kernel<float>), rgrid, rblock, 0, p.stream, planes, parts, count,
                                   static_cast<float*>(p.y));
            else
                hipLaunchKernelGGL((parts_reduce_kernel<_Float16>), rgrid, rblock, 0, p.stream, planes, parts, count,
                                   static_cast<_Float16*>(p.y));
            return hipGetLastError();
        }
    }
    if (p.out == OutType::F32)
        hipLaunchKernelGGL((prefill_ring_kernel<TM, WN, GATE_UP, false, float>), grid, block, 0, p.stream, x, wg, wu,
                           static_cast<float*>(p.y), static_cast<float*>(nullptr), p.M, p.N, p.K, m_tiles, n_tiles,
                           part_pairs, total, per_xcd);
    else
        hipLaunchKernelGGL((prefill_ring_kernel<TM, WN, GATE_UP, false, _Float16>), grid, block, 0, p.stream, x, wg, wu,
                           static_cast<_Float16*>(p.y), static_cast<float*>(nullptr), p.M, p.N, p.K, m_tiles, n_tiles,
                           part_pairs, total, per_xcd);
    return hipGetLastError();
}

}  // namespace

// K a multiple of 256 (rows start on 16 bytes, whole super-pairs) below 2^20
// (32-bit offsets inside a tile), every operand 16-byte aligned.
bool prefill_ring_supports(const Problem& p) {
    const auto on16 = [](const void* v) { return (reinterpret_cast<uintptr_t>(v) & 15u) == 0; };
    return p.K % 256 == 0 && p.K > 0 && p.K < (1u << 20) && on16(p.x) && on16(p.w) && on16(p.w_up);
}

// Where K is long and the tiles are few, K parts of 128-row tiles fill the chip:
// the least of rounds of one workgroup per CU x (5 us + super-pairs of a part x
// their time) + reduction, against 95 % of a bm x bn tiling's own rounds less 0.4
// us per part (with 92 % and nothing per part, 65 x 4096 x 4096 took 20.0 us
// instead of 17.0 and 64 x 3072 x 2048 15.3 instead of 13.7; of 303 shapes that took
// parts then none is slower than its own tiles now).  Fits to
// MI355X timings in us per super-pair: 3.6 (128 x 256), 2.2 (128 x 128), the
// staging-wave tiles 1.25 (64 x 128), 0.85 (64 x 64); the reduction 3 us and the
// planes written and read once at 4 TB/s, planes up to 48 MiB (inside a
// library stream's prompt scratch).  Measured against the tiles it
// replaced (us): 128 / 256 x 14 336 x 4096 51.0 -> 30.1, 56.3 -> 43.2; 400 x 14
// 336 x 5120 118 -> 82; 100 x 13 824 x 5120 49.4 -> 31.7; 65 x 28 672 x 8192 114
// -> 73; 32 x 11 008 x 4096 39.4 -> 22.8.
hipError_t launch_prefill_ring_parts(const Problem& p, int bm, int bn) {
    const double cus = kquant::device_cus();
    const uint32_t nsuper = p.K / 256u;
    auto cost = [&](int tm, int tn, double each, uint32_t parts) {
        const double tiles = static_cast<double>((p.M + tm - 1u) / tm) * ((p.N + tn - 1u) / tn) * parts;
        double us = std::ceil(tiles / cus) * (5.0 + each * ((nsuper + parts - 1) / parts));
        if (parts > 1) us += 3.0 + 8.0 * p.M * p.N * parts / 4e6;
        return us;
    };
    const double own = cost(bm, bn, bm == 128 ? (bn == 256 ? 3.6 : 2.2) : (bn == 128 ? 1.25 : 0.85), 1);
    double best = own;
    int tile = 0;
    uint32_t parts = 1;
    for (int tn = 256; tn >= 128; tn /= 2)
        for (uint32_t k = 2; k <= 8 && k * 2 <= nsuper + 1; ++k) {
            if (4.0 * p.M * p.N * k > 48.0 * 1048576.0) break;
            const double us = cost(128, tn, tn == 256 ? 3.6 : 2.2, k);
            if (us < best) {
                best = us;
                tile = tn;
                parts = k;
            }
        }
    if (tile == 0 || best + 0.4 * parts >= 0.95 * own) return hipErrorNotSupported;
    return tile == 256 ? launch_ring<4, 4, false>(p, parts) : launch_ring<4, 2, false>(p, parts);
}

// The rings fill and drain once per tile: with short K the staging-wave body of
// the same tiles is the faster one.  Linear, this body against it in us: 65 x 256 x
// 28 672 10.2 / 7.5, 100 x 1024 x 28 672 16.2 / 14.6, 256 x 1536 x 14 336 20.1 /
// 19.5, 65 x 2048 x 28 672 23.7 / 22.9; from 2048 with more than one row of tiles it
// gains (1 to 3 % on average there, 4 % at 4096).  Gate/up (less to hand over): 2048
// x 768 x 28 672 287 / 260, 80 x 768 x 28 672 19.6 / 18.7; on average 1 % faster at
// 1024, 2 to 4 % from 2048.
bool prefill_ring_pays(const Problem& p, bool gate_up) {
    return p.K >= (gate_up ? 1024u : p.M > 128 ? 2048u : 2304u);
}

hipError_t launch_prefill_ring(const Problem& p, int bm, int bn, bool gate_up, uint32_t parts) {
    if (bm != 128) return hipErrorInvalidValue;
    if (gate_up) return bn == 128 && parts == 1 ? launch_ring<4, 4, true>(p, 1) : hipErrorInvalidValue;
    return bn == 256   ? launch_ring<4, 4, false>(p, parts)
           : bn == 128 ? launch_ring<4, 2, false>(p, parts)
                       : hipErrorInvalidValue;
}

}  // namespace mote::q4_0
