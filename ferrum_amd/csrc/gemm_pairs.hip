// Projection of a batch of f32 rows, Y[M,N] = X[M,K] . W[N,K]^T for Q4_K / Q5_K / Q6_K / IQ4_XS weights, on the f16
// matrix instruction, no farther from 64 bits than on the f32 one: neither side is rounded to 16 bits.
//
// * A weight of these formats is a block scale times an integer (less dmin times an integer).  sc * (q - 8) of Q4_K and
//   sc * (q - 16) of Q5_K have at most ten bits and are exact f16 values; sc * (q - 32) of Q6_K and ls * codebook of
//   IQ4_XS have up to thirteen and travel as their f16 rounding and the exact remainder.  The block scale d is applied
//   to the f32 sums of a super-block.
// * An activation is two f16 values: x * s = hi + lo, s a power of two per row and super-block that brings the largest
//   to [2^14, 2^15).  hi and lo carry 23 bits and the sign between them: five elements of six are exact, the others off by
//   their last bit (2^-23 of the element at most, 0.6 2^-24 in the mean square; below 2^-15 of the largest one 2^-39 of that).
// * What the centring by 8 or 16 leaves, sum over the eight groups of (centre * d * sc - dmin * m) * (sum of x), is
//   four steps of the f32 matrix instruction per super-block, on group sums taken in f64.
// * The sums of the super-blocks are added in f64 (and, where a weight has two parts, their pieces too), which pays for
//   the operands' last bits.  rel-L2 to 64 bits in 1e-7, f32 instruction / f32 sums here / this, 24 x 5120 x 17408 Q6_K:
//   normal rows 1.19 / 1.15 / 0.78, SiLU times up 1.18 / 1.25 / 0.92, a channel in 250 a thousand times the others
//   1.17 / 1.36 / 1.08; Q4_K 1.19 / 1.07 / 0.85, 1.18 / 1.12 / 0.91, 1.18 / 1.21 / 1.01.  The projections of a layer of
//   24 rows take 106.7 us, with f32 sums 106.4.
//
// The rows are split once per call by split_rows_kernel, into the order in which a wave reads matrix operands, so the
// product itself has no conversion of activations.  The alternative, v_mfma_f32_16x16x4_f32 on exact f32 weights
// (gemm_rows.hpp, which keeps smaller matrices and Q8_0), does a sixteenth of the work per instruction and decodes
// every weight once per 16 rows.
//
// What bounds it: the waves' own instructions.  24 x 28672 x 4096 takes 37 us; with no weight or operand on its way in the
// loop 30, also without decode 29, with half the multiplications 28: eight waves a compute unit (136 KB of operands, 222 -
// 247 registers) do not hide the vector instructions of one behind the matrix instructions of another as four would.
//
// A workgroup is eight waves: two halves of K (every other super-block) x four tiles of 32 weight rows; all 32 rows of
// the batch's group at once.  A super-block's operands are brought into LDS by LDS-direct loads one super-block ahead
// and shared by the four waves of a K half; every wave requests its own raw weights two super-blocks ahead into
// registers.
#include <algorithm>

#include "device_utils.hpp"
#include "internal.hpp"
#include "lds_direct.hpp"
#include "tile_decode.hpp"

namespace fh {
namespace {

typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));   // native vectors: a value stays one run of registers

constexpr uint32_t kGroupRows = 32;                  // rows of the batch a workgroup multiplies
constexpr uint32_t kTileRows = 32;                   // weight rows of a wave
constexpr uint32_t kTileWaves = 4, kHalves = 2;
constexpr uint32_t kThreads = 64 * kTileWaves * kHalves;
constexpr uint32_t kWorkgroupRows = kTileRows * kTileWaves;
// operands of one super-block of one group: hi (16 steps x 64 lanes x 16 bytes), lo, the group sums (4 steps x 64 lanes
// x 4 bytes), 32 inverse scales, rounded up to a kilobyte
constexpr uint32_t kLoAt = 16384, kSumsAt = 32768, kInverseAt = 33792, kOperandBytes = 34816;

// ---- the rows, split ---------------------------------------------------------------------

template <int CTRL>
__device__ __forceinline__ double lane_swap(double v) {
    const uint64_t bits = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)bits, CTRL, 0xf, 0xf, false);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(bits >> 32), CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// Weights of a super-block in operand order: lane half K / 128, step 4 * (K / 32 % 4) + K / 8 % 4, and within the eight
// of a step and lane 0 2 1 3 4 6 5 7: the order in which masked quant dwords give them.
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ x, uint8_t* __restrict__ out, uint32_t m,
                                                         uint32_t nb) {
    constexpr uint32_t kRows = 2;   // a wave's: the launch is a few round trips long whatever it moves
    const uint32_t lane = threadIdx.x & 63u, wave = blockIdx.z * 4 + (threadIdx.x >> 6), b = blockIdx.x, group = blockIdx.y;
    uint8_t* const base = out + ((size_t)group * nb + b) * kOperandBytes;
    float4 v[kRows];
#pragma unroll
    for (uint32_t i = 0; i < kRows; ++i) {
        const uint32_t row = group * kGroupRows + wave * kRows + i;
        v[i] = row < m ? *reinterpret_cast<const float4*>(x + ((size_t)row * nb + b) * 256 + 4 * lane)
                       : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (uint32_t i = 0; i < kRows; ++i) {
        const uint32_t row = wave * kRows + i;   // of the group
        const float e[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
        uint32_t most = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) most = max(most, __float_as_uint(e[j]) & 0x7fffffffu);
        const bool has_nan = __ballot(most > 0x7f800000u) != 0;
        most = __float_as_uint(wave_max(__uint_as_float(min(most, 0x7f800000u))));   // (NaN counts as an infinity)
        // (a super-block with an infinity or a NaN has no such scale: it counts as zeros and an infinite or NaN inverse,
        // either of which makes the sum NaN: resolve_nan)
        const bool finite = most < 0x7f800000u;
        const uint32_t exponent = min(max(268u - (most >> 23), 1u), 253u);
        const float s = __uint_as_float(exponent << 23), inverse = __uint_as_float((254u - exponent) << 23);
        uint32_t hi[4], lo[4];
        double sum = 0.0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float scaled = finite ? e[j] * s : 0.f;
            hi[j] = f32_to_f16_bits(scaled);
            lo[j] = f32_to_f16_bits(scaled - f16_bits_to_f32(hi[j]));
            sum += (double)scaled;
        }
        const uint32_t at = (((lane >> 3) & 3u) * 4 + ((lane & 7u) >> 1)) * 1024 + (row + 32 * (lane >> 5)) * 16 + 8 * (lane & 1u);
        *reinterpret_cast<uint2*>(base + at) = make_uint2(hi[0] | (hi[2] << 16), hi[1] | (hi[3] << 16));
        *reinterpret_cast<uint2*>(base + kLoAt + at) = make_uint2(lo[0] | (lo[2] << 16), lo[1] | (lo[3] << 16));
        sum += lane_swap<0xB1>(sum);    // quad_perm [1,0,3,2]
        sum += lane_swap<0x4E>(sum);    // quad_perm [2,3,0,1]
        sum += lane_swap<0x141>(sum);   // row_half_mirror: the other quad of each 8
        const uint32_t g = lane >> 3;   // the sum of group g = 4 h + i belongs to lane half h, step i
        if ((lane & 7u) == 0)
            *reinterpret_cast<float*>(base + kSumsAt + (g & 3u) * 256 + (row + 32 * (g >> 2)) * 4) = (float)sum;
        if (lane == 0)
            *reinterpret_cast<float*>(base + kInverseAt + 4 * row) =
                finite ? inverse : __uint_as_float(has_nan ? 0x7fc00000u : 0x7f800000u);
    }
}

// ---- raw weights of one lane: half a super-block (128 weights) of one row -------------------

__device__ __forceinline__ half2v as_half2(uint32_t v) { return __builtin_bit_cast(half2v, v); }
__device__ __forceinline__ half2v twice(float v) { return half2v{(_Float16)v, (_Float16)v}; }

// The compiler waits for what a load brings here at the latest (and counts it as waited for from then on).
template <class Loaded>
__device__ __forceinline__ void landed(Loaded& v) {
    asm volatile("" : "+v"(v));
}

__device__ __forceinline__ u32x4 load_u32x4_unaligned(const uint8_t* p) {
    u32x4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}

constexpr float kTwoTo14 = 16384.f, kTwoTo16 = 65536.f;

// Interface of a format: load(block, h) requests half h (weights 128 h ..) and wait() waits for it; unpack(h) sets up the scales;
// step<S>(first, rest) gives the eight weights of step S as f16 integers times 2^-14 (kScale undoes it, with d) and,
// where kParts is 2, the remainders of their rounding; offset(i) is the exact f32 factor of the sum of x over group
// 4 h + i.
template <uint32_t TYPE>
struct Half;

template <bool FIFTH>
struct KQuants {   // Q4_K, Q5_K
    static constexpr uint32_t kBlockBytes = FIFTH ? 176 : 144;
    static constexpr int kLoads = FIFTH ? 7 : 5, kParts = 1;
    static constexpr bool kOffset = true;
    u32x4 hdr, q[4], high[FIFTH ? 2 : 1];
    float d, off[4];
    half2v a[4], b[4];
    __device__ __forceinline__ void load(const uint8_t* block, uint32_t h) {
        hdr = *reinterpret_cast<const u32x4*>(block);
        if constexpr (FIFTH) {
            high[0] = *reinterpret_cast<const u32x4*>(block + 16);
            high[1] = *reinterpret_cast<const u32x4*>(block + 32);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = *reinterpret_cast<const u32x4*>(block + (FIFTH ? 48 : 16) + 64 * h + 16 * i);
    }
    __device__ __forceinline__ void wait() {
        landed(hdr);
        if constexpr (FIFTH) landed(high[0]), landed(high[1]);
#pragma unroll
        for (int i = 0; i < 4; ++i) landed(q[i]);
    }
    __device__ __forceinline__ void unpack(uint32_t h) {
        constexpr float kCentre = FIFTH ? 16.f : 8.f;
        const float dmin = f16_bits_to_f32(hdr.x >> 16), d0 = f16_bits_to_f32(hdr.x & 0xffffu);
        d = d0 * kTwoTo14;
        // scales and minimums of groups 4 h .. 4 h + 3, a byte each
        const uint32_t upper = 0u - h;
        const uint32_t sc = (((hdr.w & 0x0f0f0f0fu) | ((hdr.y >> 2) & 0x30303030u)) & upper) | (hdr.y & 0x3f3f3f3fu & ~upper);
        const uint32_t mn = ((((hdr.w >> 4) & 0x0f0f0f0fu) | ((hdr.z >> 2) & 0x30303030u)) & upper) |
                            (hdr.z & 0x3f3f3f3fu & ~upper);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float s = (float)((sc >> (8 * i)) & 0xffu), m = (float)((mn >> (8 * i)) & 0xffu);
            // a masked low nibble reads as q 2^-24, a high one as 16 q 2^-24
            a[i] = twice((i & 1) ? s * 64.f : s * 1024.f);
            b[i] = twice(s * (-kCentre / kTwoTo14));
            off[i] = fmaf(kCentre * d0, s, -(dmin * m));
        }
        if constexpr (FIFTH) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                high[i].x >>= 4 * h;
                high[i].y >>= 4 * h;
                high[i].z >>= 4 * h;
                high[i].w >>= 4 * h;
            }
        }
    }
    template <int S>
    __device__ __forceinline__ void step(uint4& first, uint4&) const {
        constexpr int slice = S / 4, u = S % 4;   // slice: 32 weights of chunk slice / 2, low or high nibbles
        const u32x4& from = q[2 * (slice / 2) + u / 2];
        uint32_t out[4];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint32_t w = (u & 1) ? (j ? from.w : from.z) : (j ? from.y : from.x);
            constexpr uint32_t mask = (slice & 1) ? 0x00f000f0u : 0x000f000fu;
            uint32_t q02 = w & mask, q13 = (w >> 8) & mask;
            if constexpr (FIFTH) {
                const u32x4& bits = high[u / 2];
                const uint32_t p = (u & 1) ? (j ? bits.w : bits.z) : (j ? bits.y : bits.x);
                constexpr int up = (slice & 1) ? 8 : 4;
                q02 |= (p << (up - slice)) & (0x00010001u << up);
                constexpr int down = 8 - (up - slice);
                q13 |= (p >> down) & (0x00010001u << up);
            }
            out[2 * j] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(as_half2(q02), a[slice], b[slice]));
            out[2 * j + 1] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(as_half2(q13), a[slice], b[slice]));
        }
        first = make_uint4(out[0], out[1], out[2], out[3]);
    }
};
template <>
struct Half<kQ4K> : KQuants<false> {};
template <>
struct Half<kQ5K> : KQuants<true> {};

// A centred quant (an exact f16 subnormal) times its scale: the rounding and what it leaves, both exact f16 values.
__device__ __forceinline__ void scaled_parts(half2v centred, half2v scale, uint32_t& rounded, uint32_t& rest) {
    const half2v r = centred * scale;
    rounded = __builtin_bit_cast(uint32_t, r);
    rest = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(centred, scale, -r));
}

template <>
struct Half<kQ6K> {
    static constexpr uint32_t kBlockBytes = 210;
    static constexpr int kLoads = 8, kParts = 2;
    static constexpr bool kOffset = false;
    u32x4 low[4], plane[2];
    u32x2 sc;
    uint32_t dh;
    float d, off[1];
    half2v a[8];
    __device__ __forceinline__ void load(const uint8_t* block, uint32_t h) {
#pragma unroll
        for (int i = 0; i < 4; ++i) low[i] = load_u32x4_unaligned(block + 64 * h + 16 * i);
        plane[0] = load_u32x4_unaligned(block + 128 + 32 * h);
        plane[1] = load_u32x4_unaligned(block + 144 + 32 * h);
        __builtin_memcpy(&sc, block + 192 + 8 * h, 8);
        dh = load_u16_unaligned(block + 208);
    }
    __device__ __forceinline__ void wait() {
#pragma unroll
        for (int i = 0; i < 4; ++i) landed(low[i]);
        landed(plane[0]), landed(plane[1]);
        landed(sc), landed(dh);
    }
    __device__ __forceinline__ void unpack(uint32_t) {
        d = f16_bits_to_f32(dh) * kTwoTo16;   // (scales of up to 128: the integers travel as multiples of 2^-16)
#pragma unroll
        for (int i = 0; i < 8; ++i) {   // scale i: slice i / 2, positions 16 (i % 2) ..
            const float s = (float)(int)(int8_t)((i < 4 ? sc.x : sc.y) >> (8 * (i & 3)));
            a[i] = twice(i < 4 ? s * 256.f : s * 16.f);
        }
    }
    template <int S>
    __device__ __forceinline__ void step(uint4& first, uint4& rest) const {
        constexpr int slice = S / 4, u = S % 4;
        constexpr bool upper = slice >= 2;   // high nibbles, four bits up in place
        const u32x4& from = low[2 * (slice & 1) + u / 2];
        const u32x4& bits = plane[u / 2];
        const half2v centre = twice(upper ? -512.f / 16777216.f : -32.f / 16777216.f);
        uint32_t o[4], r[4];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint32_t w = (u & 1) ? (j ? from.w : from.z) : (j ? from.y : from.x);
            const uint32_t p = (u & 1) ? (j ? bits.w : bits.z) : (j ? bits.y : bits.x);
            constexpr uint32_t mask = upper ? 0x00f000f0u : 0x000f000fu, two = upper ? 0x03000300u : 0x00300030u;
            constexpr int left = (upper ? 8 : 4) - 2 * slice;   // 4, 2, 4, 2
            const uint32_t q02 = (w & mask) | ((p << left) & two), q13 = ((w >> 8) & mask) | ((p >> (8 - left)) & two);
            scaled_parts(as_half2(q02) + centre, a[2 * slice + u / 2], o[2 * j], r[2 * j]);
            scaled_parts(as_half2(q13) + centre, a[2 * slice + u / 2], o[2 * j + 1], r[2 * j + 1]);
        }
        first = make_uint4(o[0], o[1], o[2], o[3]);
        rest = make_uint4(r[0], r[1], r[2], r[3]);
    }
};

template <>
struct Half<kIQ4XS> {
    static constexpr uint32_t kBlockBytes = 136;
    static constexpr int kLoads = 5, kParts = 2;
    static constexpr bool kOffset = false;
    u32x2 hdr;
    u32x4 q[4];
    float d, off[1];
    half2v a[4];
    __device__ __forceinline__ void load(const uint8_t* block, uint32_t h) {
        hdr = *reinterpret_cast<const u32x2*>(block);
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = load_u32x4_unaligned(block + 8 + 64 * h + 16 * i);
    }
    __device__ __forceinline__ void wait() {
        landed(hdr);
#pragma unroll
        for (int i = 0; i < 4; ++i) landed(q[i]);
    }
    __device__ __forceinline__ void unpack(uint32_t h) {
        d = f16_bits_to_f32(hdr.x & 0xffffu) * kTwoTo14;
        const uint32_t low = hdr.y >> (16 * h), high = hdr.x >> (16 + 8 * h);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t ls = ((low >> (4 * i)) & 15u) | (((high >> (2 * i)) & 3u) << 4);
            a[i] = twice((float)((int)ls - 32) * 1024.f);
        }
    }
    template <int S>
    __device__ __forceinline__ void step(uint4& first, uint4& rest) const {
        constexpr int slice = S / 4, u = S % 4;   // u = 0, 1: low nibbles of two dwords, 2, 3: high nibbles
        const half2v centre = twice(-128.f / 16777216.f);
        uint32_t o[4], r[4];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const u32x4& from = q[slice];
            const uint32_t w = ((u & 1) ? (j ? from.w : from.z) : (j ? from.y : from.x)) >> (u >= 2 ? 4 : 0);
            const uint32_t bytes = iq4_lookup4(w);
            const uint32_t q02 = bytes02_as_halves(bytes), q13 = bytes13_as_halves(bytes);
            scaled_parts(as_half2(q02) + centre, a[slice], o[2 * j], r[2 * j]);
            scaled_parts(as_half2(q13) + centre, a[slice], o[2 * j + 1], r[2 * j + 1]);
        }
        first = make_uint4(o[0], o[1], o[2], o[3]);
        rest = make_uint4(r[0], r[1], r[2], r[3]);
    }
};

// ---- the product ---------------------------------------------------------------------------

struct PairsParams {
    const uint8_t* w;
    const uint8_t* operands;   // [groups][nb][kOperandBytes]
    const float* x;            // the rows themselves
    void* y;
    uint32_t m, n, nb, y_dtype;
    uint32_t groups, tile_groups, segments, seg_blocks;
    float* partials;           // [segments][m][n]
    uint32_t* counters;        // one per (tile group, group), zero between launches
};

__device__ __forceinline__ float16v mfma_f16(uint4 a, uint4 b, float16v c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
}

template <uint32_t TYPE>
__device__ __forceinline__ float weight_of(const uint8_t* w, uint32_t row, uint32_t column, uint32_t nb) {
    if constexpr (TYPE == kQ4K) return q4k_weight(w, row, column, nb);
    else if constexpr (TYPE == kQ5K) return q5k_weight(w, row, column, nb);
    else if constexpr (TYPE == kQ6K) return q6k_weight(w, row, column, nb);
    else return iq4xs_weight(w, row, column, nb);
}

// A wave's sums that are NaN, for a row of the batch with infinities but no NaN (x, and its inverse scales, which say
// which super-blocks have them): the products of the infinities and the lane's weight row are what decides.  `sum` is 0, or NaN where the
// weights themselves have a scale that is not finite.  Over as soon as every lane has met a NaN (infinities of both
// signs, or one times a weight of zero).
template <uint32_t TYPE>
__device__ __attribute__((noinline)) float infinite_products(const uint8_t* w, const float* x, const uint8_t* inverse, uint32_t row,
                                                             uint32_t nb, float sum) {
    const uint32_t lane = threadIdx.x & 63u;
    for (uint32_t b0 = 0; b0 < nb; b0 += 64) {
        const float f = *reinterpret_cast<const float*>(inverse + (size_t)min(b0 + lane, nb - 1) * kOperandBytes);
        uint64_t blocks = __ballot(b0 + lane < nb && __builtin_isinf(f));
        for (; blocks != 0; blocks &= blocks - 1) {
            const uint32_t b = b0 + (uint32_t)__builtin_ctzll(blocks);
            const float4 v = *reinterpret_cast<const float4*>(x + (size_t)b * 256 + 4 * lane);
            const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                uint64_t lanes = __ballot(__builtin_isinf(e[j]));
                for (; lanes != 0; lanes &= lanes - 1) {
                    const uint32_t from = (uint32_t)__builtin_ctzll(lanes);
                    sum = fmaf(weight_of<TYPE>(w, row, b * 256 + 4 * from + j, nb), __shfl(e[j], (int)from, 64), sum);
                    if (__ballot(sum == sum) == 0) return sum;
                }
            }
        }
    }
    return sum;
}

// The sums of a wave, COUNT a lane, where one is NaN: v[i] of lane half kg belongs to row first(i) + kg * step of the
// group.  Rows with a NaN keep it; rows with infinities get their products' sum; any other NaN (a scale of the weights, an overflow
// in both directions) stays.  24 x 5120 x 17408 Q6_K, us: finite rows 52, NaN rows 57, one infinity 95, one in every row 132,
// all of every row 180.  (Multiplying a row out again, value by value, took 4 ms, for all rows 65.)
template <uint32_t TYPE, int COUNT, class First>
__device__ __forceinline__ void resolve_nan(const PairsParams& p, float (&v)[COUNT], uint32_t group, uint32_t row, First&& first,
                                            uint32_t step) {
    uint64_t any = 0;
#pragma unroll
    for (int i = 0; i < COUNT; ++i) any |= __ballot(v[i] != v[i]);
    if (any == 0) return;
    const uint32_t lane = threadIdx.x & 63u, kg = lane >> 5;
    const uint8_t* const inverse = p.operands + (size_t)group * p.nb * kOperandBytes + kInverseAt;
    bool nan = false, infinite = false;   // of row lane % 32, every other super-block
    for (uint32_t b = kg; b < p.nb; b += 2) {
        const float f = *reinterpret_cast<const float*>(inverse + (size_t)b * kOperandBytes + 4 * (lane & 31u));
        nan = nan || f != f;
        infinite = infinite || __builtin_isinf(f);
    }
    const uint64_t nans = __ballot(nan), infinities = __ballot(infinite);
    const uint32_t rows = ((uint32_t)infinities | (uint32_t)(infinities >> 32)) & ~((uint32_t)nans | (uint32_t)(nans >> 32));
    if (rows == 0) return;
    const uint32_t weight_row = min(row, p.n - 1);
    float zero = 0.f;
    for (uint32_t b = 0; b < p.nb; ++b) zero = fmaf(weight_of<TYPE>(p.w, weight_row, b * 256, p.nb), 0.f, zero);
#pragma unroll
    for (int i = 0; i < COUNT; ++i) {
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
            const uint32_t t = first(i) + h * step;
            if ((rows >> t & 1u) == 0) continue;
            const float sum = infinite_products<TYPE>(p.w, p.x + (size_t)(group * kGroupRows + t) * p.nb * 256, inverse + 4 * t, weight_row,
                                                      p.nb, zero);
            if (kg == h) v[i] = sum;
        }
    }
}

template <uint32_t TYPE>
__global__ __launch_bounds__(kThreads) void gemm_pairs_kernel(const PairsParams p) {
    using Raw = Half<TYPE>;
    constexpr uint32_t kBB = Raw::kBlockBytes;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ uint32_t last_flag;

    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t half = wave / kTileWaves, tile_wave = wave % kTileWaves;
    const uint32_t r32 = lane & 31u, kg = lane >> 5;

    // XCD x takes the x-th eighth of the items (segment, tile group, row group), row groups fastest: those of a tile
    // group share its weights in that XCD's L2
    uint32_t group, tile_group, segment;
    {
        const uint32_t items = p.groups * p.tile_groups * p.segments, xcd = blockIdx.x & 7u, at = blockIdx.x >> 3;
        const uint32_t begin = (uint32_t)((uint64_t)items * xcd >> 3), end = (uint32_t)((uint64_t)items * (xcd + 1) >> 3);
        if (begin + at >= end) return;
        const uint32_t item = begin + at, column = item / p.groups;
        group = item - column * p.groups;
        segment = column / p.tile_groups;
        tile_group = column - segment * p.tile_groups;
    }
    const uint32_t row0 = tile_group * kWorkgroupRows + tile_wave * kTileRows, row = row0 + r32;
    const uint32_t first_block = segment * p.seg_blocks, blocks = min(p.seg_blocks, p.nb - first_block);
    const uint32_t mine = (blocks - half + kHalves - 1) / kHalves;   // of this half

    // rows past the matrix re-read its last one; what they produce is never stored
    const uint8_t* const wrow = p.w + ((size_t)min(row, p.n - 1) * p.nb + first_block + half) * kBB;
    const uint8_t* const operands = p.operands + ((size_t)group * p.nb + first_block + half) * kOperandBytes;
    uint8_t* const slots = lds + half * 2 * kOperandBytes;

    // A super-block's operands: 32 kilobytes of hi and lo, eight to a wave, and one more instruction a wave for the last
    // two kilobytes (two waves each repeat one, with the same bytes, so that all waves count the same loads).  The
    // compiler does not see these loads (it would wait for them before any read of LDS); the wait at the head of a round
    // covers them.
    const uint32_t slots_at = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)slots);
    auto request = [&](uint32_t i) {
        const uint8_t* const src = operands + (size_t)i * kHalves * kOperandBytes;
        const uint32_t dst = slots_at + (i & 1u) * kOperandBytes;
#pragma unroll
        for (uint32_t j = 0; j < 9; ++j) {
            const uint32_t at = 1024 * (j < 8 ? 4 * j + tile_wave : 32 + (tile_wave & 1u));
            lds_load16_at(src + at, 16 * lane, dst + at);
        }
    };

    double acc[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.0;

    Raw raw[2];
    if (mine > 0) {
        raw[0].load(wrow, kg);
        __builtin_amdgcn_sched_barrier(0);
        request(0);
        __builtin_amdgcn_sched_barrier(0);
        raw[1].load(wrow + (size_t)(mine > 1 ? 1 : 0) * kHalves * kBB, kg);
        __builtin_amdgcn_sched_barrier(0);
    }
    auto round = [&](uint32_t i, Raw& here, auto in_loop) {
        constexpr bool kLoop = decltype(in_loop)::value;
        // This round's operands, and the weights requested before them, have landed once no more than the weight
        // requests behind them are outstanding (loads retire in order); the build counts those in the generated code.
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoop ? Raw::kLoads : 0) : "memory");
        __syncthreads();   // ... in every wave, and the other slot has been read by all
        here.wait();       // ahead of the next requests, which the compiler cannot count
        __builtin_amdgcn_sched_barrier(0);
        if (kLoop || i + 1 < mine) request(min(i + 1, mine - 1));
        __builtin_amdgcn_sched_barrier(0);
        here.unpack(kg);
        const uint8_t* const slot = slots + (i & 1u) * kOperandBytes;
        // (the large products in chains of eight or four steps: with all sixteen in one the product was as far from 64
        // bits as on the f32 instruction, Q6_K and IQ4_XS farther)
        constexpr int kChains = Raw::kParts == 2 ? 4 : 2;
        float16v hi[kChains], lo, sums;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            lo[v] = sums[v] = 0.f;
#pragma unroll
            for (int c = 0; c < kChains; ++c) hi[c][v] = 0.f;
        }
        auto steps = [&](auto self, auto at) {
            constexpr int s = decltype(at)::value;
            if constexpr (s < 16) {
                uint4 first, rest;
                here.template step<s>(first, rest);
                const uint4 xh = *reinterpret_cast<const uint4*>(slot + 1024 * s + 16 * lane);
                const uint4 xl = *reinterpret_cast<const uint4*>(slot + kLoAt + 1024 * s + 16 * lane);
                hi[s * kChains / 16] = mfma_f16(xh, first, hi[s * kChains / 16]);
                lo = mfma_f16(xl, first, lo);
                if constexpr (Raw::kParts == 2) {
                    lo = mfma_f16(xh, rest, lo);
                    lo = mfma_f16(xl, rest, lo);
                }
                self(self, std::integral_constant<int, s + 1>{});
            }
        };
        steps(steps, std::integral_constant<int, 0>{});
        if constexpr (Raw::kOffset) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const float xs = *reinterpret_cast<const float*>(slot + kSumsAt + 256 * s + 4 * lane);
                sums = __builtin_amdgcn_mfma_f32_32x32x2f32(xs, here.off[s], sums, 0, 0, 0);
            }
        }
        const float d = here.d;
        if constexpr (kLoop)   // (past the last super-block that one again: the counts stay the same)
            here.load(wrow + (size_t)min(i + 2, mine - 1) * kHalves * kBB, kg);
        // element v of a lane: row 8 (v / 4) + 4 kg + v % 4 of the group, weight row r32
#pragma unroll
        for (int v4 = 0; v4 < 4; ++v4) {
            const float4 inv = *reinterpret_cast<const float4*>(slot + kInverseAt + 32 * v4 + 16 * kg);
            const float scale[4] = {inv.x, inv.y, inv.z, inv.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int v = 4 * v4 + j;
                if constexpr (kChains == 4) {
                    const double sum = ((double)hi[0][v] + (double)hi[1][v]) + ((double)hi[2][v] + (double)hi[3][v]) + (double)lo[v];
                    acc[v] = fma(sum, (double)(d * scale[j]), acc[v]);
                } else {
                    const float sum = hi[0][v] + hi[1][v] + lo[v];
                    acc[v] = fma((double)fmaf(d, sum, sums[v]), (double)scale[j], acc[v]);
                }
            }
        }
    };
    // (two rounds of both halves at a time and no way past either: the compiler's own counts of outstanding loads are
    // exact then, and its waits for one set of weights leave the other, and the operands, on their way)
    constexpr std::true_type loop{};
    constexpr std::false_type last{};
    const uint32_t common = blocks / kHalves;
    const bool odd = blocks % kHalves != 0;   // a last super-block of the first half's
    uint32_t i = 0;
    for (; i + 2 <= common; i += 2) {
        round(i, raw[0], loop);
        round(i + 1, raw[1], loop);
    }
    if (i < common) {
        round(i, raw[0], last);
        if (odd) {
            if (half == 0) round(i + 1, raw[1], last);
            else __syncthreads();
        }
    } else if (odd) {
        if (half == 0) round(i, raw[0], last);
        else __syncthreads();
    }

    // the two halves of K meet in LDS
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    double2* const exchange = reinterpret_cast<double2*>(lds) + (size_t)tile_wave * 512 + lane;
    if (half == 1) {
#pragma unroll
        for (int v = 0; v < 8; ++v) exchange[64 * v] = make_double2(acc[2 * v], acc[2 * v + 1]);
    }
    __syncthreads();
    const uint32_t m0 = group * kGroupRows;
    if (half == 0) {
        float sum[16];
#pragma unroll
        for (int v = 0; v < 8; ++v) {
            const double2 other = exchange[64 * v];
            sum[2 * v] = (float)(acc[2 * v] + other.x);
            sum[2 * v + 1] = (float)(acc[2 * v + 1] + other.y);
        }
        if (p.segments == 1) resolve_nan<TYPE>(p, sum, group, row, [](int v) { return (uint32_t)(8 * (v / 4) + v % 4); }, 4);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const uint32_t token = m0 + 8 * (v / 4) + 4 * kg + v % 4;
            if (row < p.n && token < p.m) {
                if (p.segments == 1)
                    store_from_f32(p.y, (size_t)token * p.n + row, p.y_dtype, sum[v]);
                else   // device scope: coherent across the chip's L2 slices without cache-wide flushes
                    __hip_atomic_store(p.partials + ((size_t)segment * p.m + token) * p.n + row, sum[v], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
    if (p.segments == 1) return;
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the stores above have completed
    __syncthreads();
    if (tid == 0) {
        uint32_t* const counter = p.counters + tile_group * p.groups + group;
        const uint32_t ticket = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t last = ticket == p.segments - 1 ? 1u : 0u;
        if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last_flag = last;
    }
    __syncthreads();
    if (last_flag == 0) return;
    // the last workgroup to arrive adds the segments in order; both halves of it, sixteen rows each, four segments of
    // eight outputs on their way at a time (one load after the other took longer than the product)
    double total[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) total[j] = 0.0;
    const float* const from = p.partials + min(row, p.n - 1);
    for (uint32_t s0 = 0; s0 < p.segments; s0 += 4) {
        float part[4][8];
#pragma unroll
        for (uint32_t s = 0; s < 4; ++s)
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) {
                const uint32_t token = min(m0 + 16 * half + 2 * j + kg, p.m - 1);
                part[s][j] = __hip_atomic_load(from + ((size_t)min(s0 + s, p.segments - 1) * p.m + token) * p.n, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
            }
#pragma unroll
        for (uint32_t s = 0; s < 4; ++s)
            if (s0 + s < p.segments) {
#pragma unroll
                for (uint32_t j = 0; j < 8; ++j) total[j] += (double)part[s][j];
            }
    }
    float sum[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) sum[j] = (float)total[j];
    resolve_nan<TYPE>(p, sum, group, row, [half](int j) { return 16 * half + 2 * (uint32_t)j; }, 1);
#pragma unroll
    for (uint32_t j = 0; j < 8; ++j) {
        const uint32_t token = m0 + 16 * half + 2 * j + kg;
        if (row < p.n && token < p.m) store_from_f32(p.y, (size_t)token * p.n + row, p.y_dtype, sum[j]);
    }
}

template <uint32_t TYPE>
void launch_one(hipStream_t s, const PairsParams& p) {
    constexpr size_t kLds = kHalves * 2 * kOperandBytes;
    static std::atomic<uint64_t> raised{0};
    once_per_device(raised, [] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_pairs_kernel<TYPE>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds);
    });
    const uint32_t items = p.groups * p.tile_groups * p.segments;
    hipLaunchKernelGGL((gemm_pairs_kernel<TYPE>), dim3((items + 7) / 8 * 8), dim3(kThreads), kLds, s, p);
}

}  // namespace

// Against the f32 matrix instruction (profiles/f32_batches_pairs_us.txt; us, that / this; 24 rows Q4_K 28672 x 4096 117 / 37, 5120 x 17408 86 / 35, 34816 x 5120
// 148 / 69, 4096 x 4096 21.4 / 19.4; Q6_K 4096 x 14336 65 / 41).  A launch of this kernel and the one that splits the rows
// take 16 us however small the matrix, and up to 16 rows half of the 32 it multiplies are empty, so those go by format:
// 16 rows Q4_K 17408 x 5120 48 / 38, 5120 x 5120 20.1 / 20.5, 4096 x 4096 12 / 19, Q5_K 6144 x 6144 25.2 / 24.4, 7147 x 4352
// 20.6 / 22.3, Q6_K 34816 x 5120 97 / 125.  Rows of one or two super-blocks leave one K half of a workgroup idle or both with a
// single round: 8 x 126084 x 256 Q4_K 18.3 / 22.5, 14 x 76728 x 512 Q5_K 24.1 / 28.5 and even at 300,000 super-blocks; of three
// 10 x 50643 x 768 Q4_K 31.6 / 21.4.  33 to 48
// rows are two groups here and three there: 48 rows Q4_K 5120 x 5120 36 / 30, 4096 x 4096 30 / 31, Q6_K 5120 x 5120 44 / 47,
// 6144 x 6144 73 / 55.
bool pairs_pay(uint32_t ggml_type, uint32_t n, uint32_t k, uint32_t m) {
    const uint64_t blocks = (uint64_t)n * (k / 256);
    if (ggml_type == kQ8_0 || m < 7 || n < 2560) return false;
    if (m <= 16) return k > 512 && ((ggml_type == kQ4K && blocks >= 120000u) || (ggml_type == kQ5K && blocks >= 140000u));
    if (m > 32 && m <= 48) return blocks >= (ggml_type == kQ6K ? 131072u : 100000u);
    return blocks >= 65536u;
}

RowsPlan gemm_pairs_plan(uint32_t n, uint32_t k, uint32_t m, int cu_count) {
    RowsPlan plan{};
    const uint32_t nb = k / 256, cus = cu_count > 0 ? (uint32_t)cu_count : 256u;
    plan.pairs = true;
    plan.rows = kGroupRows;
    plan.k_waves = kHalves;
    plan.tiles = kTileRows / 16;
    plan.tile_groups = (n + kWorkgroupRows - 1) / kWorkgroupRows;
    // K segments, from the matrix alone: the sums of a row then do not depend on how many rows come with it
    double best = 1e300;
    for (uint32_t segments = 1; segments <= 16; ++segments) {
        const uint32_t seg_blocks = (nb + segments - 1) / segments;
        if ((nb + seg_blocks - 1) / seg_blocks != segments || (segments > 1 && seg_blocks < 2)) continue;
        const uint64_t wgs = (uint64_t)plan.tile_groups * segments;
        const double us = (double)((wgs + cus - 1) / cus) * (4.0 + 3.2 * ((seg_blocks + 1) / 2)) + (segments > 1 ? 6.0 : 0.0);
        if (us < best) {
            best = us;
            plan.segments = segments;
            plan.seg_blocks = seg_blocks;
        }
    }
    // groups of a launch: their operands and partial sums fit the scratch a device has at all times
    const size_t operands = (size_t)nb * kOperandBytes;
    const size_t sums = plan.segments > 1 ? (size_t)plan.segments * n * sizeof(float) * kGroupRows : 0;
    uint64_t most = fh_device::kScratchFloor / (operands + sums);
    if (plan.segments > 1) most = std::min<uint64_t>(most, fh_device::kCounterWords / plan.tile_groups);
    most = std::min<uint64_t>(std::max<uint64_t>(most, 1), 65535u);
    plan.run_rows = (uint32_t)std::min<uint64_t>(m, most * kGroupRows);
    plan.groups = (plan.run_rows + kGroupRows - 1) / kGroupRows;
    plan.counters = plan.segments > 1 ? (size_t)plan.tile_groups * plan.groups : 0;
    plan.operand_bytes = operands * plan.groups;
    plan.partial_bytes = plan.operand_bytes + (plan.segments > 1 ? (size_t)plan.segments * plan.run_rows * n * sizeof(float) : 0);
    return plan;
}

void launch_gemm_pairs(hipStream_t s, const GemmArgs& a) {
    const RowsPlan& plan = a.rows_plan;
    PairsParams p{};
    p.w = static_cast<const uint8_t*>(a.w);
    p.operands = reinterpret_cast<const uint8_t*>(a.partials);
    p.partials = reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(a.partials) + plan.operand_bytes);
    p.counters = a.counters;
    p.n = a.n;
    p.nb = a.k / 256;
    p.y_dtype = a.y_dtype;
    p.tile_groups = plan.tile_groups;
    p.segments = plan.segments;
    p.seg_blocks = plan.seg_blocks;
    const size_t y_row = (size_t)a.n * dtype_bytes(a.y_dtype);
    for (uint32_t first = 0; first < a.m; first += plan.run_rows) {
        p.x = static_cast<const float*>(a.x) + (size_t)first * a.k;
        p.y = static_cast<uint8_t*>(a.y) + first * y_row;
        p.m = std::min(plan.run_rows, a.m - first);
        p.groups = (p.m + kGroupRows - 1) / kGroupRows;
        hipLaunchKernelGGL(split_rows_kernel, dim3(p.nb, p.groups, kGroupRows / 8), dim3(256), 0, s, p.x,
                           const_cast<uint8_t*>(p.operands), p.m, p.nb);
        switch (a.ggml_type) {
            case kQ4K: launch_one<kQ4K>(s, p); break;
            case kQ5K: launch_one<kQ5K>(s, p); break;
            case kQ6K: launch_one<kQ6K>(s, p); break;
            default: launch_one<kIQ4XS>(s, p); break;
        }
    }
}

}  // namespace fh
