// K-quant (and Q8_0) linear over many tokens on the matrix cores, y[M, N] = x[M, K] (f16)
// . W[N, K]^T with Q4_K or Q6_K weights (layouts in kquant.hip).
//
// A workgroup of 4 x 2 waves computes a 32 TM x 128 tile of y over one part of
// K.  Wave (kg, wn) owns 32 weight rows (columns 32 wn .. of the tile) for
// group kg's share of the part's super-blocks, TM tiles of
// v_mfma_f32_32x32x16_f16 with the activations as the A operand.  Lane (r, c)
// (r = lane % 32, c = lane / 32) supplies weight row r and, in the slice
// (h, u) of quarter p of a super-block, its elements
//   64 p + 32 h + 16 c + 8 u .. + 7,
// so a lane's quants of a quarter are contiguous bytes: it loads them itself,
// global memory to registers, half a super-block at a time, and re-uses the
// registers for the same half of the next super-block as soon as they are
// decoded (two to three quarters ahead of their use; no LDS traffic for the
// weights).
//
// Weight operands are exact binary16 integers, as in the few-token tiles of
// kquant.hip: Q4_K sc q (at most 63 x 15), one packed fma from 1024 + q or 64 +
// q; Q6_K sc (q - 32) = 8 s (q - 32) + t (q - 32) with s = sc >> 3, t = sc & 7,
// two operands (q - 32) s and (q - 32) t / 8 into the same accumulator.  Every
// product with an activation is exact in f32; once per super-block
//   Q4_K: y += d C - dmin C',  C' = sum_j m_j S_j (two bfloat16 MFMAs: S_j, the
//         f32 sum of the activations over sub-block j, in three pieces, exact
//         and of any size, against m_j)
//   Q6_K: y += 8 d C.
// So the decode costs 10 (Q4_K) or 20 (Q6_K) vector instructions per 8
// weights and TM MFMAs (2 TM for Q6_K), and the per-super-block fold 16 TM.
//
// Activations: direct-to-LDS 16-byte loads, 64 k of every group per interval,
// four slots (three intervals in flight while one is multiplied), 128-byte rows
// with the 16-byte chunks XOR-swizzled by half the row: the 16 rows that an
// operand read covers per cycle fall on the 64 banks once (swizzled by the row,
// every read took 8 cycles instead of 4).  One barrier per interval, before its last slice:
// the slice's MFMAs cover the first LDS reads and decode of the next interval.
// The Q4_K sums come through LDS too (kq_sums_kernel writes them before), one
// super-block ahead: as binary16 hi + lo loaded to registers they made sums
// past 65504 recompute the token's outputs one by one, and the 128-row tile
// spilled and waited for every load in flight once per super-block (512 x 4096
// x 14 336 83.9 us against 81.7, 256 x 14 336 x 4096 47.6 against 46.9).
//
// The groups' partial tiles meet in LDS (fixed order); K parts, used where the
// tiles are too few for the chip, meet in scratch planes that
// parts_reduce_kernel adds in part order.  Planes and sums live in the stream's
// prompt scratch (q4_0.hpp).  Without it there is one part, and Q4_K's sums are
// added up from the operands in registers, 16 elements per lane, three MFMAs per
// super-block (OWN): 32 dot products per tile and quarter in every wave, which 96-
// and 64-row tiles have registers for.  512 x 4096 x 14 336 121 us against 80, 256 x 14 336 x 4096 92
// against 46.
//
// A result that is not finite is added up again with GGML's values, over the
// activations and blocks that make it so (over all elements, as in the few-token
// tiles, 300 x 4096 x 4096 Q4_K with NaN activations took 64 ms and with one
// infinite activation in each token as long, now 0.16 and 2.2 ms).
//
// Measured on MI355X (weights of three calls rotated): 512 x 4096 x 14 336 Q4_K
// 80 us (750 TFLOP/s), where the four-token passes of the LDS-ring GEMV, which
// read every weight M / 4 times, took 1723; 256 x 14 336 x 4096 Q6_K 62 us
// against 1203.  Bound by the interval's instruction stream: counters have MFMAs
// in 37 (Q4_K) and 44 % (Q6_K) of all SIMD cycles and 7.0 and 5.4 vector
// instructions per MFMA, imperfectly overlapped at two waves per SIMD.  96- and
// 64-row tiles take 8 and 20 % longer per row and are for token counts and grids
// that 128-row tiles fill badly (300 x 4096 x 14 336: 65 us on 96-row tiles).
// Activations off the 16-byte grid, and such Q4_K weights, keep the kernels of
// few tokens in passes.  The Q8_0 linear has a kernel of its own
// (q8_0_prefill_ring.hpp) and shares the launch.
#include "export.hpp"
#include "kquant_blocks.hpp"
#include "q4_0.hpp"
#include "q8_0_prefill_ring.hpp"
#include "tile_ops.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace mote::kquant {
namespace {

// 16-byte vector at a 2-byte-aligned address (one unaligned dwordx4 load).
typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));

constexpr int kTileWaves = 4;   // waves along N
constexpr int kTileGroups = 2;  // groups of them along K

// Keeps a converted scale in f32: as mixed-precision fmas from the binary16
// word, two of which in a row need a wait state, the folds took twice as long.
__device__ __forceinline__ float as_f32(float v) {
    asm("" : "+v"(v));
    return v;
}

// A lane's quants of one super-block and the words its scales come from.
template <Fmt F>
struct Raw;
template <>
struct Raw<Fmt::Q4K> {
    u32x4 qs[4];  // bytes 16 c .. 16 c + 15 of quarter p's 32
    u32x4 head;   // d, dmin, scales
};
template <>
struct Raw<Fmt::Q6K> {
    u32x4 la[2], lb[2], qh[2];  // per half block: ql bytes 16 c.. of its two 32-byte runs, qh bytes 16 c..
    u32x4 sc;
    uint32_t d;
};


// The scales of the super-block being multiplied.
template <Fmt F>
struct Scales;

template <>
struct Scales<Fmt::Q4K> {
    uint32_t sc[2];  // sc_0..3, sc_4..7, a byte each
    uint32_t m[4];   // m_0, m_1; .. m_6, m_7 as bfloat16
    float d, dmin;
};
template <>
struct Scales<Fmt::Q6K> {
    uint32_t sc[4];  // quarter p: its scales at bytes 0 (h = 0) and 2 (h = 1)
    float d;
};

// The row's sum of GGML's values where it is not finite, one thread: it is the
// sum over the activations that are not finite and the blocks of such scales.
template <Fmt F>
__device__ inline float kq_not_finite_thread(const uint8_t* row, const uint16_t* xrow, uint32_t nb) {
    auto special = [](uint32_t half) { return (half & 0x7C00u) == 0x7C00u; };
    float acc = 0.0f;
    for (uint32_t b = 0; b < nb; ++b, row += block_bytes<F>()) {
        const auto* at = reinterpret_cast<const uint16_t*>(row);
        const bool scale = F == Fmt::Q4K ? special(at[0]) || special(at[1]) : special(at[104]);
        for (uint32_t c = 0; c < kSuper; c += 8, xrow += 8) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(xrow);
            const uint32_t u[4] = {v.x, v.y, v.z, v.w};
            bool any = scale;
#pragma unroll
            for (int i = 0; i < 4; ++i) any |= special(u[i]) || special(u[i] >> 16);
            if (!any) continue;
            for (uint32_t e = 0; e < 8; ++e)
                if (scale || special(xrow[e])) acc += half_bits_to_float(xrow[e]) * kq_value<F>(row, c + e);
            if (acc != acc) return acc;
        }
    }
    return acc;
}

// A float as three bfloat16 (eight significant bits each, cut off: exact).
struct Pieces {
    uint32_t p[3];
};
__device__ __forceinline__ Pieces pieces(float v) {
    const uint32_t a = __builtin_bit_cast(uint32_t, v) & 0xFFFF0000u;
    const float r = v - __builtin_bit_cast(float, a);
    const uint32_t b = __builtin_bit_cast(uint32_t, r) & 0xFFFF0000u;
    const uint32_t c = __builtin_bit_cast(uint32_t, r - __builtin_bit_cast(float, b));
    return {{a >> 16, b >> 16, c >> 16}};
}
// Two bytes of w, at selectors a and b, as a pair of bfloat16.
template <int A, int B>
__device__ __forceinline__ uint32_t bytes_bf16(uint32_t w) {
    const float a = static_cast<float>((w >> (8 * A)) & 0xFFu), b = static_cast<float>((w >> (8 * B)) & 0xFFu);
    return perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07060302u);
}

// OWN (Q4_K): each wave adds up the sub-blocks' activations itself instead of
// reading kq_sums_kernel's.
template <Fmt F, int TM, bool SK, typename OutT, bool OWN = false>
__global__ __launch_bounds__(64 * kTileWaves * kTileGroups) void kq_prefill_kernel(
    const uint16_t* __restrict__ x, const uint8_t* __restrict__ w, const uint16_t* __restrict__ sums,
    OutT* __restrict__ y, float* __restrict__ partial, uint32_t M, uint32_t N, uint32_t K, uint32_t m_tiles,
    uint32_t n_tiles, uint32_t part_blocks, uint32_t total, uint32_t per_xcd) {
    constexpr int KG = kTileGroups;
    constexpr int BM = 32 * TM;
    constexpr uint32_t BN = 32 * kTileWaves;
    constexpr int kUnit = BM * 128;            // LDS bytes of one group's activations of an interval
    constexpr int kSlots = 4;                  // interval t, a quarter p = t % 4 of a super-block: slot p
    constexpr int NA = BM / (8 * kTileWaves);  // activation loads per wave and interval
    constexpr int NB = F == Fmt::Q6K ? 2 : 1;  // operands per 8 weights
    // Block sums: the 64-row Q6_K tiles, which also serve few tokens, keep the
    // two operands' sums apart (half as many roundings in a row: 1.2e-7 of the
    // result at K = 4096, as the few-token tiles, against 1.45e-7).
    constexpr int NC = NB == 2 && TM == 2 ? 2 : 1;
    // ... and add up the result in runs of kRun super-blocks, then the runs:
    // a single chain over one K part of 56 super-blocks was coarser than the
    // few-token tiles' sixteen waves (64 x 14 336 x 32 768 Q4_K 1.68e-7 of the
    // result against 1.35e-7, Q6_K 1.36e-7 against 1.28e-7; in runs 1.32e-7 and
    // 1.17e-7, at the same time).
    constexpr bool RUNS = TM == 2;
    constexpr uint32_t kRun = 8;
    constexpr uint32_t BB = block_bytes<F>();
    constexpr int kRing = kSlots * KG * kUnit;
    // The activations' sums: 64 bytes per row, two super-blocks of each group.
    constexpr bool SUMS = F == Fmt::Q4K && !OWN;
    constexpr int NS = SUMS ? (BM * 64 + kTileWaves * 1024 - 1) / (kTileWaves * 1024) : 0;  // loads per wave
    constexpr int kSumUnit = NS * kTileWaves * 1024;
    constexpr int kReduce = kTileWaves * KG * ((TM + 1) / 2) * 4096;
    static_assert(kRing >= kReduce && kRing + 2 * KG * kSumUnit <= 160 * 1024, "LDS");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kRing + 2 * KG * kSumUnit];

    const uint32_t logical = (blockIdx.x % 8u) * per_xcd + blockIdx.x / 8u;
    if (logical >= total) return;
    const uint32_t tile_m = logical % m_tiles, rest = logical / m_tiles;
    const uint32_t tile_n = rest % n_tiles, part = rest / n_tiles;
    const uint32_t m0 = tile_m * BM, n0 = tile_n * BN;
    const uint32_t nb = K / kSuper;
    const uint32_t pb0 = part * part_blocks, pb1 = min(pb0 + part_blocks, nb);

    const int lane = static_cast<int>(threadIdx.x) & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int kg = wave / kTileWaves, wn = wave % kTileWaves;
    const int lr = lane & 31, lc = lane >> 5;
    // this group's super-blocks: [b0, b0 + ns)
    const uint32_t per = (pb1 - pb0 + KG - 1) / KG;
    const uint32_t b0 = min(pb0 + static_cast<uint32_t>(kg) * per, pb1);
    const uint32_t ns = min(per, pb1 - b0);

    // Activation load i of a wave covers 8 rows; position p of row r holds the
    // chunk (8 elements) of slice position q = p ^ (r / 2) % 8, chunk 4 h + 2 c
    // + u for q = 4 c + 2 h + u.
    const uint8_t* xb = reinterpret_cast<const uint8_t*>(x) + (static_cast<size_t>(m0) * K + b0 * kSuper) * 2;
    uint32_t aoff[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const uint32_t row = (wn * NA + i) * 8 + (lane >> 3);
        const uint32_t q = (lane & 7) ^ ((row >> 1) & 7);
        aoff[i] = (min(m0 + row, M - 1) - m0) * (K * 2) + (4 * ((q >> 1) & 1) + 2 * (q >> 2) + (q & 1)) * 16;
    }
    const Buffer xsrc = buffer_at(xb);
    uint8_t* const unit = lds + kg * kUnit;
    const uint32_t last = ns * 4 - 1;
    auto load_a = [&](uint32_t t, uint32_t slot) {  // interval t (clamped) of this group
        const uint32_t o = min(t, last) * 128u;
#pragma unroll
        for (int i = 0; i < NA; ++i)
            load_lds16(xsrc, aoff[i], o, unit + slot * (KG * kUnit) + (wn * NA + i) * 1024);
    };
    // Weights: row r of this wave's 32 (clamped), from super-block b0 on.
    const uint8_t* const wrow =
        w + (static_cast<size_t>(min(n0 + wn * 32 + lr, N - 1)) * nb + b0) * BB;
    Raw<F> raw;
    // After the second quarter of a half block, p = 1 or 3: that half's quants
    // of super-block s (clamped).  A quarter at a time, as it is freed, fetched
    // the lines of a row's half block twice.
    auto load_quants = [&](auto pc, uint32_t s) {
        constexpr int P = decltype(pc)::value, g = P / 2;
        if constexpr (P % 2 == 1) {
            const size_t at = static_cast<size_t>(min(s, ns - 1)) * BB;
            const uint8_t* blk = wrow + at;
            if constexpr (F == Fmt::Q4K) {
#pragma unroll
                for (int p = 2 * g; p < 2 * g + 2; ++p)
                    raw.qs[p] = *reinterpret_cast<const u32x4*>(blk + 16 + 32 * p + 16 * lc);
            } else {
                raw.la[g] = *reinterpret_cast<const u32x4_a2*>(blk + 64 * g + 16 * lc);
                raw.lb[g] = *reinterpret_cast<const u32x4_a2*>(blk + 64 * g + 32 + 16 * lc);
                raw.qh[g] = *reinterpret_cast<const u32x4_a2*>(blk + 128 + 32 * g + 16 * lc);
            }
        }
    };
    auto load_head = [&](uint32_t s) {
        const size_t at = static_cast<size_t>(min(s, ns - 1)) * BB;
        const uint8_t* blk = wrow + at;
        if constexpr (F == Fmt::Q4K) {
            raw.head = *reinterpret_cast<const u32x4*>(blk);
        } else {
            raw.sc = *reinterpret_cast<const u32x4_a2*>(blk + 192);
            raw.d = *reinterpret_cast<const uint16_t*>(blk + 208);
        }
    };
    Scales<F> sl;
    float d_fold = 0.0f;  // the scale of the block sums not yet folded
    auto unpack_head = [&]() {
        if constexpr (F == Fmt::Q4K) {
            const u32x4 head = raw.head;
            sl.sc[0] = head.y & 0x3F3F3F3Fu;
            sl.sc[1] = (head.w & 0x0F0F0F0Fu) | ((head.y >> 2) & 0x30303030u);
            const uint32_t lo = head.z & 0x3F3F3F3Fu;
            const uint32_t hi = ((head.w >> 4) & 0x0F0F0F0Fu) | ((head.z >> 2) & 0x30303030u);
            sl.m[0] = bytes_bf16<0, 1>(lo);
            sl.m[1] = bytes_bf16<2, 3>(lo);
            sl.m[2] = bytes_bf16<0, 1>(hi);
            sl.m[3] = bytes_bf16<2, 3>(hi);
            sl.d = as_f32(half_lo_to_float(head.x));
            sl.dmin = as_f32(half_hi_to_float(head.x));
        } else {
            const uint32_t s[4] = {raw.sc.x, raw.sc.y, raw.sc.z, raw.sc.w};
#pragma unroll
            for (int p = 0; p < 4; ++p) sl.sc[p] = s[p] >> (8 * lc);
            sl.d = as_f32(8.0f * half_bits_to_float(raw.d));
        }
    };
    // The binary16 factors of a quarter's two sub-blocks (h = 0, 1).
    f16x2 mul[2][NB], add[2][NB];
    auto quarter_scales = [&](auto pc) {
        constexpr int P = decltype(pc)::value;
        if constexpr (F == Fmt::Q4K) {
            const uint32_t word = sl.sc[P / 2];
            const f16x2 sc = as_h2(perm(0x64646464u, word, P % 2 ? 0x04030402u : 0x04010400u)) +
                             both(static_cast<_Float16>(-1024.0f));
            mul[0][0] = both(sc, false);
            mul[1][0] = both(sc, true);
            add[0][0] = mul[0][0] * both(static_cast<_Float16>(-1024.0f));
            add[1][0] = mul[1][0] * both(static_cast<_Float16>(-64.0f));
        } else {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int sc = static_cast<int8_t>((sl.sc[P] >> (16 * h)) & 0xFFu);
                const _Float16 s = static_cast<_Float16>(static_cast<short>(sc >> 3));
                const _Float16 t =
                    static_cast<_Float16>(static_cast<short>(sc & 7)) * static_cast<_Float16>(0.125f);
                mul[h][0] = both(s);
                mul[h][NB - 1] = both(t);
                add[h][0] = both(static_cast<_Float16>(s * static_cast<_Float16>(-1056.0f)));
                add[h][NB - 1] = both(static_cast<_Float16>(t * static_cast<_Float16>(-1056.0f)));
            }
        }
    };
    // The operands of slice (h, u) of quarter p.
    f16x8 b[2][NB];
    auto decode = [&](auto pc, auto uc, f16x8 (&dst)[NB]) {
        constexpr int P = decltype(pc)::value, U = decltype(uc)::value, h = U / 2, u = U % 2;
        uint32_t q[2];
        if constexpr (F == Fmt::Q4K) {
            constexpr uint32_t mask = h ? 0xF0F0F0F0u : 0x0F0F0F0Fu, e = h ? 0x54545454u : 0x64646464u;
            q[0] = (u ? raw.qs[P].z : raw.qs[P].x) & mask;
            q[1] = (u ? raw.qs[P].w : raw.qs[P].y) & mask;
            const f16x2 m = mul[h][0], a = add[h][0];
            dst[0] = join(__builtin_elementwise_fma(as_h2(perm(e, q[0], 0x04010400u)), m, a),
                          __builtin_elementwise_fma(as_h2(perm(e, q[0], 0x04030402u)), m, a),
                          __builtin_elementwise_fma(as_h2(perm(e, q[1], 0x04010400u)), m, a),
                          __builtin_elementwise_fma(as_h2(perm(e, q[1], 0x04030402u)), m, a));
        } else {
            // quarter c4 of half g: nibble c4 / 2 of run c4 % 2
            constexpr int g = P / 2, c4 = 2 * (P % 2) + h;
            const u32x4 l = c4 % 2 ? raw.lb[g] : raw.la[g];
            const uint32_t lw[2] = {u ? l.z : l.x, u ? l.w : l.y};
            const uint32_t hw[2] = {u ? raw.qh[g].z : raw.qh[g].x, u ? raw.qh[g].w : raw.qh[g].y};
            f16x2 v[4];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint32_t low = (c4 < 2 ? lw[i] : lw[i] >> 4) & 0x0F0F0F0Fu;
                const uint32_t top = c4 == 0 ? hw[i] << 4 : c4 == 1 ? hw[i] << 2 : c4 == 2 ? hw[i] : hw[i] >> 2;
                q[i] = (top & 0x30303030u) | low;
                v[2 * i] = as_h2(perm(0x64646464u, q[i], 0x04010400u));
                v[2 * i + 1] = as_h2(perm(0x64646464u, q[i], 0x04030402u));
            }
#pragma unroll
            for (int k = 0; k < NB; ++k)
                dst[k] = join(__builtin_elementwise_fma(v[0], mul[h][k], add[h][k]),
                              __builtin_elementwise_fma(v[1], mul[h][k], add[h][k]),
                              __builtin_elementwise_fma(v[2], mul[h][k], add[h][k]),
                              __builtin_elementwise_fma(v[3], mul[h][k], add[h][k]));
        }
    };

    f32x16 acc[TM], blk[NC][TM], runs[RUNS ? TM : 1];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            acc[i][r] = 0.0f;
            if constexpr (RUNS) runs[i][r] = 0.0f;
#pragma unroll
            for (int c = 0; c < NC; ++c) blk[c][i][r] = 0.0f;
        }
    const f32x16 zero = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    f16x8 a[2][TM];
    const uint32_t a_row = lr * 128, a_x = (lr >> 1) & 7;
    auto read_a = [&](uint32_t slot, int u, f16x8 (&dst)[TM]) {
        const uint8_t* base = unit + slot * (KG * kUnit) + a_row + (((4 * lc + u) ^ a_x) * 16);
#pragma unroll
        for (int i = 0; i < TM; ++i) dst[i] = *reinterpret_cast<const f16x8*>(base + i * 4096);
    };
    auto multiply = [&](auto cc) {
        constexpr int C = decltype(cc)::value;
#pragma unroll
        for (int k = 0; k < NB; ++k)
#pragma unroll
            for (int i = 0; i < TM; ++i)
                blk[k % NC][i] = mfma32(a[C][i], b[C][k], blk[k % NC][i]);
    };
    // The first slice of a super-block: the sums of the one before join the
    // result, tile by tile ahead of the tile's first product.
    auto fold = [&](int i) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float sum = NC == 2 ? blk[0][i][r] + blk[NC - 1][i][r] : blk[0][i][r];
            acc[i][r] = __builtin_fmaf(d_fold, sum, acc[i][r]);
        }
    };
    auto multiply_first = [&]() {
#pragma unroll
        for (int k = 0; k < NB; ++k)
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                if (k == 0) fold(i);
                blk[k % NC][i] = mfma32(a[0][i], b[0][k], k < NC ? zero : blk[k % NC][i]);
            }
    };
    // Q4_K's minimum term of the super-block, one tile per slice of its second
    // half.  A row's sums are four 16-byte chunks: the three bfloat16 pieces of
    // the eight sub-blocks' sums, and zeros; half wave c of the two products
    // supplies chunk c, then chunk 2 + c.  In LDS a row's chunk q is at q ^ (row / 4) % 4.
    bf16x8 sx[2][2];
    uint8_t* const sum_unit = lds + kRing + kg * kSumUnit;
    uint32_t soff[NS > 0 ? NS : 1];
    const Buffer ssrc = buffer_at(reinterpret_cast<const uint8_t*>(sums) + (static_cast<size_t>(m0) * nb + b0) * 64);
#pragma unroll
    for (int i = 0; i < NS; ++i) {
        const uint32_t at = (wn * NS + i) * 64 + lane, row = at >> 2;
        soff[i] = (min(m0 + row, M - 1) - m0) * (nb * 64) + (((at & 3) ^ ((row >> 2) & 3)) * 16);
    }
    auto load_sums = [&](uint32_t s) {
#pragma unroll
        for (int i = 0; i < NS; ++i)
            load_lds16(ssrc, soff[i], min(s, ns - 1) * 64u,
                       sum_unit + (s & 1u) * (KG * kSumUnit) + (wn * NS + i) * 1024);
    };
    auto read_sums = [&](uint32_t s, int i) {
        const uint8_t* row = sum_unit + (s & 1u) * (KG * kSumUnit) + (i * 32 + lr) * 64;
#pragma unroll
        for (int k = 0; k < 2; ++k)
            sx[i & 1][k] = *reinterpret_cast<const bf16x8*>(row + (((2 * k + lc) ^ ((lr >> 2) & 3)) * 16));
    };
    auto mins = [&]() {
        if constexpr (F == Fmt::Q4K)
            return __builtin_bit_cast(bf16x8, u32x4{sl.m[0], sl.m[1], sl.m[2], sl.m[3]});
    };
    auto minimum = [&](auto pc, auto ic, uint32_t s, auto slice) {
        constexpr int I = 4 * (decltype(pc)::value - 2) + decltype(ic)::value;
        if constexpr (SUMS) {
            if constexpr (I + 1 >= 0 && I + 1 < TM) read_sums(s, I + 1);
            if constexpr (I >= 0 && I < TM) {
                const f32x16 mn = mfma32(sx[I & 1][1], mins(), mfma32(sx[I & 1][0], mins(), zero));
                slice();
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[I][r] = __builtin_fmaf(-sl.dmin, mn[r], acc[I][r]);
            } else {
                slice();
            }
        } else {
            slice();
        }
    };
    // OWN: the lane's part of sub-block j's sum, its elements 16 c .. 16 c + 15, in
    // three pieces at j of 8 (in each c: the MFMAs add both), from the slices'
    // operands; after the last slice the minimum term of every tile.
    float run[TM];
    uint32_t own[TM][3][4];
    auto add_slice = [&](auto pc, auto ic) {
        if constexpr (OWN) {
            constexpr int P = decltype(pc)::value, S = decltype(ic)::value, h = S / 2, u = S % 2;
            const uint32_t one = 0x3C003C00u;
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const u32x4 v = __builtin_bit_cast(u32x4, a[u][i]);
                const float s = dot2(v.w, one, dot2(v.z, one, dot2(v.y, one, dot2(v.x, one, u ? run[i] : 0.0f))));
                if constexpr (u == 0) {
                    run[i] = s;
                } else {
                    const Pieces b = pieces(s);
#pragma unroll
                    for (int k = 0; k < 3; ++k) own[i][k][P] = h ? own[i][k][P] | (b.p[k] << 16) : b.p[k];
                }
            }
        }
    };
    auto own_minimum = [&]() {
        if constexpr (OWN) {
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                f32x16 mn = zero;
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const u32x4 v = {own[i][k][0], own[i][k][1], own[i][k][2], own[i][k][3]};
                    mn = mfma32(__builtin_bit_cast(bf16x8, v), mins(), mn);
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][r] = __builtin_fmaf(-sl.dmin, mn[r], acc[i][r]);
            }
        }
    };
    // Loads a wave issues behind interval t's activations of four intervals on:
    // quants, the next super-block's sums (p = 0) and header (p = 2).
    constexpr bool kQ4 = F == Fmt::Q4K;
    constexpr int kHalf = kQ4 ? 2 : 3;  // a half block's quants
    constexpr int kBehind[4] = {NS, kHalf, kQ4 ? 1 : 2, kHalf};
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;

    if (ns > 0) {  // uniform over the wave; groups without work only meet the barriers
        load_sums(0);
        order_fence();
        load_a(0, 0);
        order_fence();
        load_a(1, 1);
        order_fence();
        load_quants(I1{}, 0);
        order_fence();
        load_a(2, 2);
        order_fence();
        load_head(0);
        order_fence();
        load_a(3, 3);
        order_fence();
        load_quants(I3{}, 0);
        order_fence();
        wait_counts<vm_wait(3 * NA + (kQ4 ? 5 : 8))>();  // interval 0's activations
    }
    group_barrier();
    order_fence();
    if (ns > 0) {
        read_a(0, 0, a[0]);
        unpack_head();
        quarter_scales(I0{});
        decode(I0{}, I0{}, b[0]);
        order_fence();
        // One interval: quarter p of super-block s.
        auto interval = [&](auto pc, uint32_t s) {
            constexpr int P = decltype(pc)::value;
            using PN = std::integral_constant<int, (P + 1) & 3>;
            read_a(P, 1, a[1]);
            minimum(pc, I0{}, s, [&] {
                if constexpr (P == 0) multiply_first(); else multiply(I0{});
                add_slice(pc, I0{});
                decode(pc, I1{}, b[1]);
            });
            order_fence();
            read_a(P, 2, a[0]);
            minimum(pc, I1{}, s, [&] {
                multiply(I1{});
                add_slice(pc, I1{});
                decode(pc, I2{}, b[0]);
            });
            order_fence();
            read_a(P, 3, a[1]);
            minimum(pc, I2{}, s, [&] {
                multiply(I0{});
                add_slice(pc, I2{});
                decode(pc, I3{}, b[1]);
            });
            order_fence();
            // The next interval's activations have landed (what may be
            // outstanding is all younger), and every wave has read this one's.
            wait_counts<vm_wait(2 * NA + kBehind[(P + 1) & 3] + kBehind[(P + 2) & 3] + kBehind[(P + 3) & 3]) &
                        kLgkmWait>();
            group_barrier();
            order_fence();
            read_a((P + 1) & 3, 0, a[0]);
            load_a(4 * s + P + 4, P);
            order_fence();
            load_quants(pc, s + 1);
            if constexpr (P == 2) load_head(s + 1);
            if constexpr (P == 0) load_sums(s + 1);
            order_fence();
            minimum(pc, I3{}, s, [&] {
                multiply(I1{});
                add_slice(pc, I3{});
                if constexpr (P == 3) {
                    own_minimum();
                    d_fold = sl.d;
                    unpack_head();
                }
                quarter_scales(PN{});
                decode(PN{}, I0{}, b[0]);
            });
            order_fence();
        };
        for (uint32_t s = 0; s < ns; ++s) {
            interval(I0{}, s);
            interval(I1{}, s);
            interval(I2{}, s);
            interval(I3{}, s);
            if constexpr (RUNS) {
                if (s % kRun == kRun - 1) {
#pragma unroll
                    for (int i = 0; i < TM; ++i) {
                        runs[i] += acc[i];
                        acc[i] = zero;
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            fold(i);
            if constexpr (RUNS) acc[i] += runs[i];
        }
    }
    for (uint32_t t = ns * 4; t < per * 4; ++t) group_barrier();
    wait_counts<vm_wait(0)>();
    __syncthreads();

    // Two groups: the first keeps row tiles 0 .. H - 1, the second the others;
    // each hands over the rest.
    constexpr int H = (TM + 1) / 2;
    const int kept = kg == 0 ? H : TM - H, tile0 = kg == 0 ? 0 : H;
    float* red = reinterpret_cast<float*>(lds);
    auto slot = [&](int wv, int i, int r) { return red + ((wv * H + i) * 4 + r) * 256 + lane * 4; };
    auto give = [&](const f32x16& v, int i) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            *reinterpret_cast<f32x4*>(slot(wave, i, r)) = f32x4{v[4 * r], v[4 * r + 1], v[4 * r + 2], v[4 * r + 3]};
    };
    if (kg == 0) {
#pragma unroll
        for (int i = 0; i < TM - H; ++i)
            give(acc[H + i], i);
    } else {
#pragma unroll
        for (int i = 0; i < H; ++i) {
            give(acc[i], i);
            if (H + i < TM) acc[i] = acc[H + i];
        }
        memory_fence();  // or the compiler merges both groups' writes behind selects
    }
    __syncthreads();
    const int other = wave ^ kTileWaves;
#pragma unroll
    for (int i = 0; i < H; ++i) {
        if (i >= kept) break;  // uniform
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(slot(other, i, r));
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[i][4 * r + k] += v[k];
        }
    }
    // Lane (r, c) holds column r of each tile, rows 8 (k / 4) + 4 c + k % 4.
    const uint32_t n = n0 + wn * 32 + lr;
    if (n >= N) return;
    auto token = [&](uint32_t at) { return m0 + tile0 * 32 + (at / 16) * 32 + 8 * (at / 4 % 4) + 4 * lc + at % 4; };
    auto store = [&](uint32_t m, float v) {
        if constexpr (SK)
            partial[(static_cast<size_t>(part) * M + m) * N + n] = v;
        else
            y[static_cast<size_t>(m) * N + n] = to_out<OutT>(v);
    };
    uint32_t again = 0;
#pragma unroll
    for (int i = 0; i < H; ++i) {
        if (i >= kept) break;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const uint32_t m = token(16 * i + k);
            if (m >= M) continue;
            store(m, acc[i][k]);
            again |= not_finite(acc[i][k]) ? 1u << (16 * i + k) : 0u;
        }
    }
    for (; again != 0; again &= again - 1) {
        const uint32_t m = token(__builtin_ctz(again));
        store(m, kq_not_finite_thread<F>(w + (static_cast<size_t>(n) * nb + pb0) * BB,
                                         x + static_cast<size_t>(m) * K + static_cast<size_t>(pb0) * kSuper,
                                         pb1 - pb0));
    }
}

// sums[m][b][0..7], [8..15], [16..23]: the three pieces of the sums of token m's
// activations over the eight sub-blocks of super-block b, [24..31] zeros.  One
// thread per sub-block.
__global__ __launch_bounds__(256) void kq_sums_kernel(const uint16_t* __restrict__ x, uint16_t* __restrict__ sums,
                                                      uint64_t count) {
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= count) return;
    const u32x4* src = reinterpret_cast<const u32x4*>(x + i * 32);
    const uint32_t one = 0x3C003C00u;
    float s = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const u32x4 v = src[k];
        s = dot2(v.w, one, dot2(v.z, one, dot2(v.y, one, dot2(v.x, one, s))));
    }
    const Pieces p = pieces(s);
    uint16_t* dst = sums + (i / 8) * 32 + i % 8;
#pragma unroll
    for (int k = 0; k < 3; ++k) dst[8 * k] = static_cast<uint16_t>(p.p[k]);
    dst[24] = 0;
}

// One launch over M tokens: parts > 1 into `planes` (added by a second kernel),
// Q4_K's activation sums through `sums` or, where null, OWN (64 and 96 rows).
template <Fmt F, int TM, typename OutT>
hipError_t launch_tile(const uint16_t* x, const uint8_t* w, OutT* y, uint32_t M, uint32_t N, uint32_t K,
                       uint32_t parts, float* planes, uint16_t* sums, hipStream_t stream) {
    const uint32_t nb = K / kSuper;
    const uint32_t m_tiles = (M + 32 * TM - 1) / (32 * TM), n_tiles = (N + 32 * kTileWaves - 1) / (32 * kTileWaves);
    const uint32_t part_blocks = (nb + parts - 1) / parts;
    parts = (nb + part_blocks - 1) / part_blocks;
    const uint64_t total64 = static_cast<uint64_t>(m_tiles) * n_tiles * parts;
    if (total64 > 0x7ffffff0ull) return hipErrorInvalidConfiguration;
    const uint32_t total = static_cast<uint32_t>(total64), per_xcd = (total + 7) / 8;
    if (sums != nullptr) {
        const uint64_t subs = static_cast<uint64_t>(M) * nb * 8;
        hipLaunchKernelGGL(kq_sums_kernel, dim3(static_cast<uint32_t>((subs + 255) / 256)), dim3(256), 0, stream, x,
                           sums, subs);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    const dim3 grid(per_xcd * 8), block(64 * kTileWaves * kTileGroups);
    if (parts == 1) {
        if constexpr (F == Fmt::Q8) {
            hipLaunchKernelGGL((q8_prefill_kernel<TM, false, OutT>), grid, block, 0, stream, x, w, y, planes, M, N, K,
                               m_tiles, n_tiles, part_blocks, total, per_xcd);
            return hipGetLastError();
        } else {
            if constexpr (F == Fmt::Q4K) {
                if (sums == nullptr) {
                    if constexpr (TM < 4)
                        hipLaunchKernelGGL((kq_prefill_kernel<F, TM, false, OutT, true>), grid, block, 0, stream, x, w,
                                           sums, y, planes, M, N, K, m_tiles, n_tiles, part_blocks, total, per_xcd);
                    else
                        return hipErrorInvalidValue;
                    return hipGetLastError();
                }
            }
            hipLaunchKernelGGL((kq_prefill_kernel<F, TM, false, OutT>), grid, block, 0, stream, x, w, sums, y, planes,
                               M, N, K, m_tiles, n_tiles, part_blocks, total, per_xcd);
            return hipGetLastError();
        }
    }
    if constexpr (F == Fmt::Q8)
        hipLaunchKernelGGL((q8_prefill_kernel<TM, true, float>), grid, block, 0, stream, x, w,
                           static_cast<float*>(nullptr), planes, M, N, K, m_tiles, n_tiles, part_blocks, total, per_xcd);
    else
        hipLaunchKernelGGL((kq_prefill_kernel<F, TM, true, float>), grid, block, 0, stream, x, w, sums,
                           static_cast<float*>(nullptr), planes, M, N, K, m_tiles, n_tiles, part_blocks, total, per_xcd);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const uint64_t count = static_cast<uint64_t>(M) * N;
    hipLaunchKernelGGL((parts_reduce_kernel<OutT>), dim3(parts_reduce_grid(count)), dim3(256), 0, stream, planes, parts,
                       count, y);
    return hipGetLastError();
}

// Which tile (32 tm rows) and how many K parts: the least of
//   rounds x (start + blocks x block time) + reduction,
// rounds of one workgroup per CU, blocks the super-blocks of a part, the
// reduction 3 us and the planes written and read once at 4 TB/s.  The start, 5
// us, and the block times in us are fits to MI355X timings, within 15 % at the
// shapes fitted (measured against predicted, us): Q4_K 512 x 4096 x 14 336 82 /
// 90 (128-row tiles), 101 / 109 (96-row), 99 / 113 (64-row), 100 x 4096 x 4096
// 18 / 17 (64-row, four parts); Q6_K 256 x 14 336 x 4096 88 / 102, 63 / 61
// (128-row, two, four parts); Q8_0 300 x 4096 x 14 336 80 / 93, 69 / 74, 79 / 85
// (128-, 96-, 64-row), 256 x 14 336 x 4096 52 / 53 (64-row, two parts).  Q8_0's
// 64-row tiles wait for the weights where K is long, over all of it above all: 128 x
// 8192 x 11 008 66 us, 128-row tiles over two parts 56; 512 x 11 008 x 11 008 256 and
// 203.
struct Plan {
    int tm;
    uint32_t parts;
    double us;
};
// The planes of the parts and, behind them, Q4_K's sums fill a stream's scratch.
constexpr uint64_t kMaxPlaneBytes = 48ull << 20;

// Without scratch: one part, and for Q4_K the tiles that add up the
// activations themselves (the 128-row ones would spill).
template <Fmt F>
Plan choose(uint32_t M, uint32_t N, uint32_t K, bool scratch = true) {
    const uint32_t nb = K / kSuper;
    const double cus = device_cus();
    Plan best{4, 1, 0.0};
    static constexpr double kBlockUs[3][3] = {{2.5, 1.95, 1.45}, {3.2, 2.7, 2.2}, {2.6, 2.0, 1.45}};
    for (int tm = F == Fmt::Q4K && !scratch ? 3 : 4; tm >= 2; --tm) {
        const double per_block = kBlockUs[static_cast<int>(F)][4 - tm];
        const double tiles = static_cast<double>((M + 32u * tm - 1) / (32u * tm)) * ((N + 127u) / 128u);
        for (uint32_t parts = 1; parts <= (scratch ? 8u : 1u) && parts * 2 <= nb + 1; ++parts) {
            const double plane_bytes = 4.0 * M * N * parts;
            if (parts > 1 && plane_bytes > static_cast<double>(kMaxPlaneBytes)) break;
            const double rounds = std::ceil(tiles * parts / cus);
            double block = per_block;
            if (F == Fmt::Q8 && tm == 2 && nb >= 32)
                block = parts == 1 ? 1.9 : block + 0.2 * std::min(1.0, std::max(0.0, 2.0 * tiles * parts / cus - 1.0));
            double cost = rounds * (5.0 + block * ((nb + parts - 1) / parts));
            if (parts > 1) cost += 3.0 + 2.0 * plane_bytes / 4e6;
            if (best.us == 0.0 || cost < best.us) best = {tm, parts, cost};
        }
    }
    return best;
}

// Up to 64 tokens the few-token tiles of kquant.hip compete.  Their time is
// about 4 us, 1.2 + 0.33 s (Q4_K) or 2 + 0.73 s ns per item (16 rows, 16 tokens,
// s super-blocks, at most 16), 1.9 times that with three token tiles and 1.6
// times with three K parts (256 workgroups deal those out unevenly), and 3 us
// for a part sum.  Of 1440 shapes (17 to 64 tokens, K 1024 to 16 384, N 1024 to
// 32 768) the rule slows none by more than 1.1 % against the few-token tiles;
// the largest gain it leaves is 28 %, and 64 x 14 336 x 32 768 goes from 221 (Q4_K)
// and 455 us (Q6_K) to 100 and 168.  (With a time per item that left s out, K
// below 4096 went up to 60 % slower: 32 x 1024 x 7168 Q6_K 12.9 us against 8.0, 32
// x 2048 x 20 000 Q4_K 15.3 against 13.1.)
//
// Q8_0's alternative, the tiles of q4_0_prefill.hip, is up to 12 % faster up to 64
// tokens with long K and one part, where both wait for the weights (64 x 11 008 x
// 28 672 103 us, here 115), and with K below 1024 and more than one round (512 x
// 256 x 11 008 15.2, here 17.0), but has four times the error: these serve all.
bool worth(Fmt f, uint32_t M, uint32_t N, uint32_t K) {
    if (M > 64 || f == Fmt::Q8) return true;
    if (M <= 16) return false;
    const uint32_t nb = K / kSuper, token_tiles = (M + 15) / 16, kparts = (nb + 15) / 16;
    const double items = static_cast<double>((N + 15) / 16) * token_tiles * kparts;
    const double s = nb < 16 ? nb : 16;
    double few = 4.0 + items * (f == Fmt::Q4K ? 1.2 + 0.33 * s : 2.0 + 0.73 * s) * 1e-3 *
                           (kparts == 3 ? 1.6 : token_tiles == 3 ? 1.9 : 1.0);
    if (kparts > 1) few += 3.0;
    if (0.95 * few <= 2.5 + 5.0 + 1.45) return false;  // below every plan's time
    return (f == Fmt::Q4K ? choose<Fmt::Q4K>(M, N, K) : choose<Fmt::Q6K>(M, N, K)).us + 2.5 < 0.95 * few;
}

// forced: this plan, parts 0 for one part without scratch; null: the rule's.
template <Fmt F, typename OutT>
hipError_t launch(const void* x, const void* w, void* y, uint32_t M, uint32_t N, uint32_t K, hipStream_t stream,
                  const Plan* forced = nullptr) {
    const auto* xp = static_cast<const uint16_t*>(x);
    const auto* wp = static_cast<const uint8_t*>(w);
    auto* yp = static_cast<OutT*>(y);
    auto run = [&](const Plan& p, uint32_t m0, uint32_t rows, float* planes, uint16_t* sums) {
        const uint16_t* xm = xp + static_cast<size_t>(m0) * K;
        OutT* ym = yp + static_cast<size_t>(m0) * N;
        return p.tm == 4   ? launch_tile<F, 4, OutT>(xm, wp, ym, rows, N, K, p.parts, planes, sums, stream)
               : p.tm == 3 ? launch_tile<F, 3, OutT>(xm, wp, ym, rows, N, K, p.parts, planes, sums, stream)
                           : launch_tile<F, 2, OutT>(xm, wp, ym, rows, N, K, p.parts, planes, sums, stream);
    };
    if (forced && forced->parts == 0) return run({forced->tm, 1, 0.0}, 0, M, nullptr, nullptr);
    const Plan plan = forced ? *forced : choose<F>(M, N, K);
    const uint64_t row_sums = F == Fmt::Q4K ? static_cast<uint64_t>(K / kSuper) * 64 : 0;
    if (plan.parts == 1 && row_sums == 0) return run(plan, 0, M, nullptr, nullptr);
    // Tokens whose sums do not fit beside the planes run in turns, whole tiles
    // each where that is possible.
    constexpr uint64_t kSumBytes = q4_0::kPromptScratchBytes - kMaxPlaneBytes;
    uint32_t step = M;
    if constexpr (F == Fmt::Q4K) {
        if (row_sums * M > kSumBytes) {
            step = static_cast<uint32_t>(kSumBytes / row_sums);
            if (step > 32u * plan.tm) step -= step % (32u * plan.tm);
        }
    }
    const uint64_t plane_bytes =
        plan.parts > 1 ? (static_cast<uint64_t>(step) * N * plan.parts * sizeof(float) + 15) / 16 * 16 : 0;
    q4_0::ScratchPool::Lease lease;  // holds the scratch until every kernel is queued
    const hipError_t a = q4_0::acquire_prompt_scratch(stream, plane_bytes + row_sums * step, &lease);
    if (a == hipErrorNotSupported && !forced) {
        if (M <= 64 && F != Fmt::Q8) return a;  // the kernels of few tokens
        return run(choose<F>(M, N, K, false), 0, M, nullptr, nullptr);
    }
    if (a != hipSuccess) return a;
    auto* base = static_cast<uint8_t*>(lease.ptr());
    for (uint64_t m0 = 0; m0 < M; m0 += step) {
        const hipError_t e = run(plan, static_cast<uint32_t>(m0), static_cast<uint32_t>(M - m0 < step ? M - m0 : step),
                                 reinterpret_cast<float*>(base),
                                 row_sums > 0 ? reinterpret_cast<uint16_t*>(base + plane_bytes) : nullptr);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

namespace {
bool fits(Fmt f, const void* x, const void* w, uint32_t M, uint32_t K) {
    return K % kSuper == 0 && K >= kSuper && K <= (1u << 22) && static_cast<uint64_t>(M) * (K / kSuper) <= (1ull << 31) &&
           (reinterpret_cast<uintptr_t>(x) & 15u) == 0 &&
           (reinterpret_cast<uintptr_t>(w) & (f == Fmt::Q6K ? 1u : 15u)) == 0;
}

hipError_t launch_any(Fmt f, bool f16_out, const void* x, const void* w, void* y, uint32_t M, uint32_t N, uint32_t K,
                      hipStream_t stream, const Plan* forced) {
    if (f == Fmt::Q8)
        return f16_out ? launch<Fmt::Q8, _Float16>(x, w, y, M, N, K, stream, forced)
                       : launch<Fmt::Q8, float>(x, w, y, M, N, K, stream, forced);
    if (f == Fmt::Q4K)
        return f16_out ? launch<Fmt::Q4K, _Float16>(x, w, y, M, N, K, stream, forced)
                       : launch<Fmt::Q4K, float>(x, w, y, M, N, K, stream, forced);
    return f16_out ? launch<Fmt::Q6K, _Float16>(x, w, y, M, N, K, stream, forced)
                   : launch<Fmt::Q6K, float>(x, w, y, M, N, K, stream, forced);
}
}  // namespace

bool prefill_supported(Fmt f, const void* x, const void* w, uint32_t M, uint32_t N, uint32_t K) {
    return fits(f, x, w, M, K) && worth(f, M, N, K);
}

hipError_t launch_prefill(Fmt f, bool f16_out, const void* x, const void* w, void* y, uint32_t M, uint32_t N,
                          uint32_t K, hipStream_t stream) {
    return launch_any(f, f16_out, x, w, y, M, N, K, stream, nullptr);
}

}  // namespace mote::kquant

MOTE_EXPORT int mote_hip_prompt_linear_tiles(int format, const void* input, const void* weights, void* output,
                                             uint64_t rows, uint64_t output_features, uint64_t input_features,
                                             int output_f16, int tile_rows, int k_parts, void* stream) noexcept {
    using namespace mote::kquant;
    if (!input || !weights || !output || !stream) return hipErrorInvalidValue;
    if (format != 8 && format != 12 && format != 14) return hipErrorInvalidValue;
    if (tile_rows != 64 && tile_rows != 96 && tile_rows != 128) return hipErrorInvalidValue;
    const Fmt f = format == 8 ? Fmt::Q8 : format == 12 ? Fmt::Q4K : Fmt::Q6K;
    if (k_parts < 0 || (k_parts == 0 && f == Fmt::Q4K && tile_rows == 128)) return hipErrorInvalidValue;
    if (rows == 0 || output_features == 0 || rows > UINT32_MAX || output_features > UINT32_MAX / rows ||
        input_features > (1u << 22))
        return hipErrorInvalidValue;
    const auto M = static_cast<uint32_t>(rows), N = static_cast<uint32_t>(output_features);
    const auto K = static_cast<uint32_t>(input_features);
    if (!fits(f, input, weights, M, K) || static_cast<uint32_t>(k_parts) > K / kSuper) return hipErrorInvalidValue;
    try {
        const Plan plan{tile_rows / 32, static_cast<uint32_t>(k_parts), 0.0};
        return static_cast<int>(launch_any(f, output_f16 != 0, input, weights, output, M, N, K,
                                           static_cast<hipStream_t>(stream), &plan));
    } catch (...) {
        return hipErrorUnknown;
    }
}
