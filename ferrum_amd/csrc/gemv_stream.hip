// Streamed Q4_K and Q6_K GEMV for gfx950: y[n] = sum_k W[n,k] x[k], one activation row per grid.z entry.
//
// Same product as q4_k_gemv_factored / q4_k_gemv_ksplit of the reference
// (src/metal/shaders/ops.metal:983-1070; Q6_K: q6_k_factored_rows, q6_k_gemv_ksplit and
// q6_k_gemv_factored, :1393-1439) in a form built around what limits a
// GEMV of this size on this chip: how the bytes are requested, and how few vector
// instructions are spent per weight.
//
// Bytes.  A workgroup owns up to 16 consecutive weight rows for the whole K.  Its
// waves copy those rows into LDS with LDS-direct loads (global_load_lds_dwordx4):
// every instruction moves one contiguous kilobyte of one row, nothing passes through
// registers, and all of a tile's loads are in flight before anything else happens.
//
// Arithmetic.  The nibbles never become floats on the vector ALU.  Masked in place
// inside a 16-bit half a nibble is the f16 subnormal q * 2^-24 (q * 2^-20 for a high
// nibble), which is a legal matrix-core operand, so the integer dot products
// sum q*x of every 32-weight group run on v_mfma_f32_16x16x32_f16:
//   * B operand (columns n = the tile's 16 weight rows): lane (n, g) holds eight
//     weights of chunk g (64 weights, two groups) of row n's super-block.
//   * A operand (rows j): the activations, as f16 "hi" and "lo" parts of x * s (s a
//     power of two that brings the largest magnitude of its 64-weight chunk to
//     [2^14, 2^15); hi + lo carries 22 bits; the scale is per 64-weight chunk).  Row j = 4g + i is non-zero only in
//     the k slots lane group g covers, so D[4g + i][n] is the dot product of chunk g
//     alone: i = 0 / 1 the hi / lo part against the low nibbles' group, i = 2 / 3
//     against the high nibbles' group.  Low- and high-nibble steps accumulate into
//     two D tiles; each lane (n, g) then finds the four sums of its own chunk in its
//     own registers.
//   * Per super-block a lane applies the two 6-bit scales and minimums of its chunk
//     and the block's d and dmin once.
// Q6_K quants are bytes and go to v_mfma_i32_16x16x64_i8 against four 8-bit digits of 30-bit fixed-point activations
// (stage_block_q6k): four matrix instructions per super-block where f16 parts of nibbles and bit planes took sixteen, some
// 100 vector instructions for 180, and sums of integers in place of sums over f16 subnormals: rel-L2 to 64 bits
// 0.9 - 1.1e-7, as the FMA kernel's for 16-bit rows (1.6 - 2.3e-7 for f32 ones; the f16 form's was 1e-6).  Cold,
// 151936 x 5120 145 -> 134 us, 128256 x 4096 103 -> 97, 34816 x 5120 40.2 -> 37.4.
//
// Activations.  A super-block of a tile is multiplied by exactly one wave, so that wave
// also turns the block's activations into A operands: it requests them before the
// tile's loads (loads complete in issue order, so they can be waited for with the tile
// still in flight), and passes each block through a 1 KB slot of its own in LDS, which
// re-orders the values from "four consecutive per lane" to operand order.
#include <type_traits>

#include "device_utils.hpp"
#include "internal.hpp"
#include "lds_direct.hpp"

namespace fh {
namespace {

constexpr uint32_t kQ4Bytes = 144;
constexpr uint32_t kQ6Bytes = 210;
constexpr uint32_t kSlotBytes = 1024u + 64u + 16u;   // A operands, {group sum, group sum, 1/s, -} per chunk, 16 zero bytes
// Q6_K: A operands, -32 times the digit sums of every scale group, the groups' scales, 16 zero bytes
constexpr uint32_t kAux6Bytes = 256u + 64u;
constexpr uint32_t kSlot6Bytes = 1024u + kAux6Bytes + 16u;
template <uint32_t TYPE> struct StreamFormat;
template <> struct StreamFormat<kQ4K> { static constexpr uint32_t kBytes = kQ4Bytes, kSlot = kSlotBytes, kAux = 64u; };
template <> struct StreamFormat<kQ6K> { static constexpr uint32_t kBytes = kQ6Bytes, kSlot = kSlot6Bytes, kAux = kAux6Bytes; };

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

struct StreamParams {
    const uint8_t* w;     // [n, nb] super-blocks
    const void* x;        // [m, 256 nb]
    void* y;              // [m, n]
    uint32_t n, nb;
    uint32_t tile_rows;   // rows per workgroup, 1..16
    uint32_t row_stride;  // bytes between rows of the tile in LDS
    uint32_t tile_bytes;  // of the tile region in LDS
    uint32_t x_dtype, y_dtype;
    // rows longer than a tile can hold: grid.y K segments of seg_blocks super-blocks each
    uint32_t segments, seg_blocks, m;
    uint32_t depth;       // the ring's tiles in LDS
    float* partials;      // [segments][m][n]
    uint32_t* counters;   // one per (row tile, batch row), zero between launches
};

__device__ __forceinline__ uint32_t pack_halves(_Float16 lo, _Float16 hi) {
    typedef _Float16 half2t __attribute__((ext_vector_type(2)));
    half2t v = {lo, hi};
    return __builtin_bit_cast(uint32_t, v);
}

typedef _Float16 half2v __attribute__((ext_vector_type(2)));

// f16(a s) and f16(b s) in the two halves of a dword, and f16(a s - hi) and f16(b s - hi) against such
// a pair: one v_fma_mix per value, written straight into its half (s is a power of two, so a s is
// exact and the first is the plain rounding of the product).
__device__ __forceinline__ uint32_t hi_pair(float a, float b, float s) {
    uint32_t r;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(r) : "v"(a), "v"(s));
    asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(r) : "v"(b), "v"(s));
    return r;
}
__device__ __forceinline__ uint32_t lo_pair(float a, float b, float s, uint32_t hi) {
    uint32_t r;
    asm("v_fma_mixlo_f16 %0, %1, %2, -%3 op_sel_hi:[0,0,1]" : "=v"(r) : "v"(a), "v"(s), "v"(hi));
    asm("v_fma_mixhi_f16 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "+v"(r) : "v"(b), "v"(s), "v"(hi));
    return r;
}

// One wave writes a super-block's activations (lane = float4 number inside the block) into its
// slot in operand order.  The 16 lanes of a DPP row hold one chunk (64 weights), which is what a
// lane group of the A operand covers, so the power-of-two scale is chosen per chunk and never
// leaves the row.
__device__ __forceinline__ void stage_block(float4 v, uint8_t* slot, uint32_t lane) {
    // the largest magnitude's exponent: magnitudes order like their bit patterns, and an unsigned
    // maximum folds into the DPP instruction itself
    uint32_t top = __float_as_uint(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    top = dpp_umax<0xB1>(top);
    top = dpp_umax<0x4E>(top);
    top = dpp_umax<0x141>(top);
    top = dpp_umax<0x140>(top);
    uint32_t e = top >> 23;
    e = e < 15u ? 15u : e > 254u ? 254u : e;
    const float s = __uint_as_float((268u - e) << 23);   // 2^(14 - exponent of the chunk's largest)
    // hi = f16(x s), lo = f16(x s - hi): each one fused multiply-add that rounds to a half
    const uint32_t h02 = hi_pair(v.x, v.z, s), h13 = hi_pair(v.y, v.w, s);
    const uint32_t l02 = lo_pair(v.x, v.z, s, h02), l13 = lo_pair(v.y, v.w, s, h13);
    // chunk g, group parity hbit, step u, half of the step
    const uint32_t g = lane >> 4, hbit = (lane >> 3) & 1u, u = (lane >> 1) & 3u;
    uint8_t* const dst = slot + ((u * 4u + g) * 4u + 2u * hbit) * 16u + 8u * (lane & 1u);
    // k slots of an operand dword pair are weights {0, 2} and {1, 3} of four consecutive ones
    *reinterpret_cast<uint2*>(dst) = make_uint2(h02, h13);
    *reinterpret_cast<uint2*>(dst + 16) = make_uint2(l02, l13);
    float sum = (v.x + v.y) + (v.z + v.w);
    sum = dpp_add<0xB1>(sum);
    sum = dpp_add<0x4E>(sum);
    sum = dpp_add<0x141>(sum);   // the eight lanes of a 32-weight group now all hold its sum
    // every lane writes (same value, same address within its group): {sum of x in the group, 1 / s}
    float* const aux = reinterpret_cast<float*>(slot + 1024u) + 4u * g;
    aux[hbit] = sum;
    aux[2] = __uint_as_float((e - 14u) << 23);
}

// A Q6_K super-block's activations (the layout src/metal/shaders/ops.metal:1397-1425 indexes) as integers.
// Weight 128 h + 32 s + 16 e + j (half h, slice s, j < 16) has its low four bits in
// nibble s / 2 of ql[64 h + 32 (s & 1) + 16 e + j] and its high two in bits 2 s of
// qh[32 h + 16 e + j]; lane group g = 2 h + e of the B operand holds those three 16-byte pieces,
// four scale groups of 16 weights.  Lane L holds activations 4 L .. 4 L + 3, so L = 32 h + 8 s + 4 e + j / 4: a
// quad of lanes is one scale group, which gets a power of two of its own: x 2^k = X, |X| < 2^30, and X = d0 + 256 d1 +
// 65536 d2 + 2^24 d3 with digits of a signed byte.  Row 4 g + i of the A operand is digit i of lane group g's sixteen
// activations, zero elsewhere, so one v_mfma_i32_16x16x64_i8 gives a lane the four exact digit sums of its scale group.
// The quants go in as 0 .. 63: the accumulator starts from -32 times the digits' plain sums.
__device__ __forceinline__ void stage_block_q6k(float4 v, uint8_t* slot, uint32_t lane) {
    uint32_t top = __float_as_uint(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    // (fmaxf drops a NaN beside a number: the comparison below is made on the bits)
    const uint32_t bits = max(max(__float_as_uint(v.x) << 1, __float_as_uint(v.y) << 1),
                              max(__float_as_uint(v.z) << 1, __float_as_uint(v.w) << 1)) >> 1;
    top = max(top, bits);
    top = dpp_umax<0xB1>(top);
    top = dpp_umax<0x4E>(top);
    const uint32_t ex = min(top >> 23, 254u);
    const int shift = 156 - (int)ex;
    const float e[4] = {v.x, v.y, v.z, v.w};
    uint32_t z[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)   // (adding 128 to the lower three digits makes them unsigned bytes; the xor takes it back)
        z[i] = ((uint32_t)(int)__builtin_ldexpf(e[i], shift) + 0x00808080u) ^ 0x00808080u;
    const uint32_t h = lane >> 5, sl = (lane >> 3) & 3u, ee = (lane >> 2) & 1u, g = 2u * h + ee;
    uint32_t* const dst = reinterpret_cast<uint32_t*>(slot + ((sl * 4u + g) * 4u) * 16u) + (lane & 3u);
    // digit i of the four, side by side
    const uint32_t a01 = __builtin_amdgcn_perm(z[1], z[0], 0x05010400u), a23 = __builtin_amdgcn_perm(z[3], z[2], 0x05010400u);
    const uint32_t b01 = __builtin_amdgcn_perm(z[1], z[0], 0x07030602u), b23 = __builtin_amdgcn_perm(z[3], z[2], 0x07030602u);
    const uint32_t digit[4] = {__builtin_amdgcn_perm(a23, a01, 0x05040100u), __builtin_amdgcn_perm(a23, a01, 0x07060302u),
                               __builtin_amdgcn_perm(b23, b01, 0x05040100u), __builtin_amdgcn_perm(b23, b01, 0x07060302u)};
    int sums[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        dst[4 * i] = digit[i];
        int t = __builtin_amdgcn_sdot4((int)digit[i], (int)0xe0e0e0e0u, 0, false);   // -32 each
        t += __builtin_amdgcn_update_dpp(0, t, 0xB1, 0xf, 0xf, false);
        t += __builtin_amdgcn_update_dpp(0, t, 0x4E, 0xf, 0xf, false);
        sums[i] = t;
    }
    // (every lane of the quad writes the same values)
    *reinterpret_cast<int4*>(slot + 1024u + (g * 4u + sl) * 16u) = make_int4(sums[0], sums[1], sums[2], sums[3]);
    // 2^(ex - 140): what undoes the shift, in units of 65536; a subnormal for the smallest.  NaN where the group has an
    // infinity or a NaN
    const uint32_t undo = top >= 0x7f800000u ? 0x7fc00000u : ex > 13u ? (ex - 13u) << 23 : 1u << (ex + 9u);
    reinterpret_cast<uint32_t*>(slot + 1024u + 256u)[g * 4u + sl] = undo;
}

// 16 or 8 bytes of a tile in LDS that are only 2-byte aligned (Q6_K blocks are 210 bytes long)
__device__ __forceinline__ uint4 lds_u4_unaligned(const uint8_t* p) {
    uint4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}
__device__ __forceinline__ uint2 lds_u2_unaligned(const uint8_t* p) {
    uint2 v;
    __builtin_memcpy(&v, p, 8);
    return v;
}

// A lane's share of one super-block, chunk g of its row against the operands of stage_block, added to acc.
__device__ __forceinline__ float multiply_q4k(const u32x4 (&xa)[4], float4 aux, uint4 hdr, uint4 qa, uint4 qb, uint32_t g, float acc) {
    const uint32_t raw[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
    floatx4 dl = {0.f, 0.f, 0.f, 0.f}, dh = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const uint32_t q0 = raw[2 * u], q1 = raw[2 * u + 1];
        const uint32_t s0 = q0 >> 8, s1 = q1 >> 8;
        const u32x4 lo = {q0 & 0x000f000fu, s0 & 0x000f000fu, q1 & 0x000f000fu, s1 & 0x000f000fu};
        const u32x4 hi = {q0 & 0x00f000f0u, s0 & 0x00f000f0u, q1 & 0x00f000f0u, s1 & 0x00f000f0u};
        const half8 a = __builtin_bit_cast(half8, xa[u]);
        dl = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, __builtin_bit_cast(half8, lo), dl, 0, 0, 0);
        dh = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, __builtin_bit_cast(half8, hi), dh, 0, 0, 0);
    }
    float sc_lo, sc_hi, mn_lo, mn_hi;
    q4k_chunk_scales(hdr.y, hdr.z, hdr.w, g, sc_lo, sc_hi, mn_lo, mn_hi);
    const float d = f16_bits_to_f32(hdr.x & 0xffffu), dmin = f16_bits_to_f32(hdr.x >> 16);
    // low nibbles were q * 2^-24, high nibbles 16 q * 2^-24
    const float dots = fmaf(sc_lo * 16777216.f, dl[0] + dl[1], (sc_hi * 1048576.f) * (dh[2] + dh[3]));
    const float mins = fmaf(mn_lo, aux.x, mn_hi * aux.y);
    return fmaf(d * aux.z, dots, fmaf(-dmin, mins, acc));
}

// The same for Q6_K: the lane group's pieces qa, qb, qh, its half's eight scales and the block's scale; dots starts
// from stage_block_q6k's sums.
__device__ __forceinline__ float multiply_q6k(const u32x4 (&xa)[4], i32x4 (&dots)[4], float4 undo, uint4 qa, uint4 qb, uint4 qh, uint2 sc8,
                                              uint16_t dbits, uint32_t e, float acc) {
    const uint32_t ql[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
    const uint32_t ph[4] = {qh.x, qh.y, qh.z, qh.w};
    i32x4 q[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        q[0][u] = (int)((ql[u] & 0x0f0f0f0fu) | ((ph[u] << 4) & 0x30303030u));
        q[1][u] = (int)((ql[4 + u] & 0x0f0f0f0fu) | ((ph[u] << 2) & 0x30303030u));
        q[2][u] = (int)(((ql[u] >> 4) & 0x0f0f0f0fu) | (ph[u] & 0x30303030u));
        q[3][u] = (int)(((ql[4 + u] >> 4) & 0x0f0f0f0fu) | ((ph[u] >> 2) & 0x30303030u));
    }
    float r[4];
    const float scale[4] = {undo.x, undo.y, undo.z, undo.w};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        dots[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, xa[t]), q[t], dots[t], 0, 0, 0);
        // a digit's sum is at most 2^16: two of them fit 32 bits and make one f32
        const float upper = (float)((dots[t][3] << 8) + dots[t][2]), lower = (float)((dots[t][1] << 8) + dots[t][0]);
        r[t] = fmaf(lower, 1.f / 65536.f, upper) * scale[t];
    }
    // the lane group's int8 scales: bytes e, e + 2, e + 4, e + 6 of its half's eight
    const uint32_t lo = sc8.x >> (8u * e), hi = sc8.y >> (8u * e);
    const float c0 = (float)(int)(int8_t)lo, c1 = (float)(int)(int8_t)(lo >> 16);
    const float c2 = (float)(int)(int8_t)hi, c3 = (float)(int)(int8_t)(hi >> 16);
    const float total = fmaf(c0, r[0], c1 * r[1]) + fmaf(c2, r[2], c3 * r[3]);
    return fmaf(f16_bits_to_f32(dbits), total, acc);
}

// LDS map (bytes): [tile: tile_rows x row_stride][a slot per wave][row sums: waves x 16 f32]
// DT: activation dtype; WAVES: waves per workgroup; MAXB: super-blocks a wave may own (row length
// <= WAVES * MAXB * 256).  Three workgroups of eight waves share a compute unit: six waves per
// SIMD (ten-wave workgroups were tried for 20-block rows, two blocks per wave; only two of them
// fit a compute unit's wave slots, and the launch took a third longer).
// OWN: a wave requests exactly the super-blocks it multiplies -- a block of all the tile's
// rows is tile_rows x 9 pieces of 16 bytes, 64 pieces per instruction -- and waits for its own
// loads only; the tile in LDS is then [block][row][144 bytes] (rows 36 words apart: sixteen rows
// read sixteen different groups of four banks).
template <uint32_t TYPE, int DT, int WAVES, int MAXB, bool OWN = false>
__device__ __forceinline__ void gemv_stream_body(const StreamParams& p) {
    constexpr uint32_t kSWaves = WAVES;
    constexpr uint32_t kBlock = StreamFormat<TYPE>::kBytes;    // bytes of a super-block
    constexpr uint32_t kSlotBytes = StreamFormat<TYPE>::kSlot;
    constexpr uint32_t kAuxBytes = StreamFormat<TYPE>::kAux;
    auto stage = [](float4 v, uint8_t* slot, uint32_t lane) {
        if constexpr (TYPE == kQ4K) stage_block(v, slot, lane);
        else stage_block_q6k(v, slot, lane);
    };
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // this workgroup's K segment: super-blocks first .. first + nb - 1 of the rows
    const uint32_t first = blockIdx.y * p.seg_blocks;
    const uint32_t nb = min(p.seg_blocks, p.nb - first);
    const uint32_t row_bytes = nb * kBlock;          // of the segment
    const uint32_t full_row_bytes = p.nb * kBlock;
    const uint32_t row0 = blockIdx.x * p.tile_rows;
    const uint32_t rows = min(p.tile_rows, p.n - row0);

    uint8_t* const tile = lds;
    uint8_t* const slot = tile + p.tile_bytes + wave * kSlotBytes;
    float* const rsum = reinterpret_cast<float*>(tile + p.tile_bytes + kSWaves * kSlotBytes);

    // 1. this wave's activation blocks are requested first.  These are register loads the
    // compiler cannot see the latency of: xraw[i] holds the data only after wait_vmcnt(issued)
    // under 3., which lets exactly the `issued` later LDS-direct loads stay in flight (vmcnt
    // retires in order, so "at most `issued` outstanding" means every load before them is done).
    // Until then nothing may read, copy or spill xraw: the empty asm with "+v"(xraw[i]) after the
    // wait is the first use the compiler is shown, the kernel has no scratch, and the build's
    // check of the generated text fails if any instruction between a load and the wait names a
    // destination register.
    const size_t xrow = ((size_t)blockIdx.z * p.nb + first) * 256u;
    typename std::conditional<DT == FH_F32, u32x4, u32x2>::type xraw[MAXB];
#pragma unroll
    for (int i = 0; i < MAXB; ++i) {
        // a wave with fewer blocks repeats its last one: the register is then defined by the
        // load alone, and nothing can touch it before the wait below
        const uint32_t b = min(wave + kSWaves * i, nb - 1u);
        // (with a scalar base and a lane offset instead of these 64-bit addresses the launch measured
        // 0.3 us slower on the 17408 x 5120 matrix, three rounds in turn on one device)
        if constexpr (DT == FH_F32) {
            const float* src = static_cast<const float*>(p.x) + xrow + b * 256u + lane * 4u;
            asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(xraw[i]) : "v"(src) : "memory");
        } else {
            const uint16_t* src = static_cast<const uint16_t*>(p.x) + xrow + b * 256u + lane * 4u;
            asm volatile("global_load_dwordx2 %0, %1, off" : "=v"(xraw[i]) : "v"(src) : "memory");
        }
    }

    // 2. the tile: instruction i covers kilobyte (i % per_row) of row (i / per_row)
    const uint32_t per_row = (row_bytes + 1023u) >> 10;
    const uint32_t total = rows * per_row;
    const uint8_t* const wbase = p.w + (size_t)row0 * full_row_bytes + (size_t)first * kBlock;
    const uint32_t tile_addr = (uint32_t)(uintptr_t)tile;
    uint32_t issued = 0;
    // OWN: a super-block of the tile is tile_rows x 9 pieces of 16 bytes, piece 64 j + lane by instruction j
    const uint32_t block_pieces = p.tile_rows * (kBlock / 16u), groups = (block_pieces + 63u) / 64u;
    const uint32_t block_pitch = block_pieces * 16u;
    if constexpr (OWN) {
        // where a lane's piece of a block lies from the block's first row on: the same for every block
        uint32_t lane_offset[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint32_t piece = 64u * j + lane, rl = piece / (kBlock / 16u), pc = piece - rl * (kBlock / 16u);
            lane_offset[j] = min(rl, rows - 1u) * full_row_bytes + 16u * pc;
        }
        const uint8_t* const first_row = p.w + (size_t)row0 * full_row_bytes + (size_t)first * kBlock;
#pragma unroll
        for (int i = 0; i < MAXB; ++i) {
            const uint32_t b = wave + kSWaves * i;
            if (b < nb) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if ((uint32_t)j < groups) {
                        if (64u * j + lane < block_pieces)
                            lds_load16_at(first_row + b * kBlock, lane_offset[j], tile_addr + b * block_pitch + 1024u * j);
                        ++issued;
                    }
                }
            }
        }
    } else {
        for (uint32_t i = wave; i < total; i += kSWaves) {
            const uint32_t r = i / per_row, c = i - r * per_row;
            if (c * 1024u + lane * 16u < row_bytes)
                lds_load16_at(wbase + (size_t)r * full_row_bytes + c * 1024u, lane * 16u,
                              tile_addr + r * p.row_stride + c * 1024u);
            ++issued;
        }
    }
    if (lane < 4u) reinterpret_cast<uint32_t*>(slot + 1024u + kAuxBytes)[lane] = 0u;

    // 3. the activations have arrived (the tile's loads may still be in flight)
    wait_vmcnt(issued);
    float4 xv[MAXB];
#pragma unroll
    for (int i = 0; i < MAXB; ++i) {
        asm volatile("" : "+v"(xraw[i])::"memory");
        if constexpr (DT == FH_F32) {
            xv[i] = make_float4(__uint_as_float(xraw[i].x), __uint_as_float(xraw[i].y), __uint_as_float(xraw[i].z),
                                __uint_as_float(xraw[i].w));
        } else if constexpr (DT == FH_F16) {
            xv[i] = make_float4(f16_bits_to_f32(xraw[i].x & 0xffffu), f16_bits_to_f32(xraw[i].x >> 16),
                                f16_bits_to_f32(xraw[i].y & 0xffffu), f16_bits_to_f32(xraw[i].y >> 16));
        } else {
            xv[i] = make_float4(bf16_bits_to_f32(xraw[i].x & 0xffffu), bf16_bits_to_f32(xraw[i].x >> 16),
                                bf16_bits_to_f32(xraw[i].y & 0xffffu), bf16_bits_to_f32(xraw[i].y >> 16));
        }
    }
    stage(xv[0], slot, lane);   // the first block while the tile is on its way
    if constexpr (!OWN) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }

    // 4. multiply this wave's super-blocks
    const uint32_t n = lane & 15u, g = lane >> 4;
    const uint32_t nc = n < rows ? n : rows - 1u;
    const bool active = (n >> 2) == g;
    const uint8_t* const wrow = tile + nc * p.row_stride;
    const uint8_t* const xlane = active ? slot + (g * 4u + (n & 3u)) * 16u : slot + 1024u + kAuxBytes;
    const uint32_t xstep = active ? 256u : 0u;
    const float* const auxp = reinterpret_cast<const float*>(slot + 1024u) + (kAuxBytes / 16u) * g;
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < MAXB; ++i) {
        const uint32_t b = wave + kSWaves * i;
        if (b < nb) {
            // this block's operands leave the slot first, so the next block can move in while
            // this one is multiplied
            u32x4 xa[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) xa[u] = *reinterpret_cast<const u32x4*>(xlane + u * xstep);
            if constexpr (OWN) {
                // this block's loads have landed when only the later blocks' are outstanding
                wait_vmcnt(issued - (uint32_t)(i + 1) * groups);
            }
            if constexpr (TYPE == kQ4K) {
                const float4 aux = *reinterpret_cast<const float4*>(auxp);
                const uint8_t* const blk = OWN ? tile + b * block_pitch + nc * kBlock : wrow + b * kBlock;
                const uint4 hdr = *reinterpret_cast<const uint4*>(blk);
                const uint4 qa = *reinterpret_cast<const uint4*>(blk + 16u + 32u * g);
                const uint4 qb = *reinterpret_cast<const uint4*>(blk + 32u + 32u * g);
                if (i + 1 < MAXB && b + kSWaves < nb) {
                    asm volatile("s_waitcnt lgkmcnt(3)" ::: "memory");   // the five slot reads are the oldest
                    stage(xv[i + 1], slot, lane);
                }
                acc = multiply_q4k(xa, aux, hdr, qa, qb, g, acc);
            } else {
                i32x4 dots[4];   // of the four scale groups, from -32 times the digits' sums
#pragma unroll
                for (int t = 0; t < 4; ++t) dots[t] = *reinterpret_cast<const i32x4*>(slot + 1024u + (g * 4u + t) * 16u);
                const float4 undo = *reinterpret_cast<const float4*>(slot + 1024u + 256u + 16u * g);
                asm volatile("" ::: "memory");   // the slot reads are issued before the tile reads
                const uint8_t* const blk = wrow + b * kBlock;
                const uint32_t h = g >> 1, e = g & 1u;
                uint4 qa, qb, qh;
                uint2 sc8;
                uint16_t dbits;
                // A read of 16 bytes that begins between two dwords takes LDS longer than the two aligned ones that cover it
                // (us: 151936 x 5120 126 / 117, 34816 x 5120 34.8 / 32.7, 5120 x 17408 22.5 / 21.5; profiles/waits_loads_lookups_us.txt).  With rows of 16 bits and two
                // blocks a wave their registers would leave two workgroups a compute unit instead of three (8192 x 28672 54 / 59).
                constexpr bool kByDwords = DT == FH_F32 || MAXB != 2;
                if (kByDwords && (b & 1u)) {   // two bytes behind a dword
                    qa = lds_u4_behind_2(blk + 64u * h + 16u * e);
                    qb = lds_u4_behind_2(blk + 64u * h + 32u + 16u * e);
                    qh = lds_u4_behind_2(blk + 128u + 32u * h + 16u * e);
                    const uint4 last = lds_u4_dword(blk + 190u + 8u * h);   // (of the second half its third dword ends the block)
                    sc8 = make_uint2(__builtin_amdgcn_alignbyte(last.y, last.x, 2), __builtin_amdgcn_alignbyte(last.z, last.y, 2));
                } else {
                    auto read = [](const uint8_t* p) { return kByDwords ? lds_u4_dword(p) : lds_u4_unaligned(p); };
                    qa = read(blk + 64u * h + 16u * e);
                    qb = read(blk + 64u * h + 32u + 16u * e);
                    qh = read(blk + 128u + 32u * h + 16u * e);
                    sc8 = lds_u2_unaligned(blk + 192u + 8u * h);
                }
                __builtin_memcpy(&dbits, blk + 208u, 2);
                if (i + 1 < MAXB && b + kSWaves < nb) {
                    // the nine slot reads are the oldest; at least five instructions read the tile
                    asm volatile("s_waitcnt lgkmcnt(5)" ::: "memory");
                    stage(xv[i + 1], slot, lane);
                }
                acc = multiply_q6k(xa, dots, undo, qa, qb, qh, sc8, dbits, e, acc);
            }
        }
    }

    // 5. chunks of a row (lanes n, n + 16, n + 32, n + 48), then the waves, in a fixed order
    acc += __shfl_xor(acc, 16, 64);
    acc += __shfl_xor(acc, 32, 64);
    if (lane < 16u) rsum[wave * 16u + lane] = acc;
    __syncthreads();
    float total_sum = 0.f;
    if (tid < rows) {
#pragma unroll
        for (int w = 0; w < kSWaves; ++w) total_sum += rsum[w * 16 + tid];
    }
    if (p.segments == 1) {
        if (tid < rows) store_from_f32(p.y, (size_t)blockIdx.z * p.n + row0 + tid, p.y_dtype, total_sum);
        return;
    }
    // 6. K segments meet in the scratch buffer and the last workgroup of a tile adds them in segment
    // order (device-scope relaxed atomics, coherent across the L2 slices; src/metal/shaders/ops.metal:1031-1070
    // has the same two-stage shape)
    const uint32_t mrow = blockIdx.z;
    if (tid < rows)
        __hip_atomic_store(&p.partials[((size_t)blockIdx.y * p.m + mrow) * p.n + row0 + tid], total_sum, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the stores above have completed
    __syncthreads();
    uint32_t* const flag = reinterpret_cast<uint32_t*>(rsum);   // the row sums have been read
    if (tid == 0) {
        uint32_t* counter = p.counters + (size_t)mrow * gridDim.x + blockIdx.x;
        const uint32_t ticket = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t last = ticket == p.segments - 1 ? 1u : 0u;
        if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *flag = last;
    }
    __syncthreads();
    if (*flag == 0) return;
    if (tid < rows) {
        float total = 0.f;
        for (uint32_t sg = 0; sg < p.segments; ++sg)
            total += __hip_atomic_load(&p.partials[((size_t)sg * p.m + mrow) * p.n + row0 + tid], __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
        store_from_f32(p.y, (size_t)mrow * p.n + row0 + tid, p.y_dtype, total);
    }
}

template <int DT, int WAVES, int MAXB>
__global__ __launch_bounds__(WAVES * kWave) __attribute__((amdgpu_waves_per_eu(6, 6)))
void gemv_stream_q4k(const StreamParams p) {
    gemv_stream_body<kQ4K, DT, WAVES, MAXB>(p);
}

template <int DT, int WAVES, int MAXB>
__global__ __launch_bounds__(WAVES * kWave) __attribute__((amdgpu_waves_per_eu(6, 6)))
void gemv_stream_q4k_own(const StreamParams p) {
    gemv_stream_body<kQ4K, DT, WAVES, MAXB, true>(p);
}

// Q6_K rows are 46% longer: two workgroups share a compute unit, four waves per SIMD.
template <int DT, int WAVES, int MAXB>
__global__ __launch_bounds__(WAVES * kWave) void gemv_stream_q6k(const StreamParams p) {
    gemv_stream_body<kQ6K, DT, WAVES, MAXB>(p);
}

// The Q4_K ring, for large matrices and one activation row: a workgroup of sixteen waves has a compute unit to itself and
// multiplies tile after tile of sixteen rows, while the next depth - 1 tiles are on their way.  With a tile per
// workgroup every sixteen rows read all activations again, turn them into operands again, and the compute
// unit asks for nothing while they multiply; here the operands of a wave's super-blocks (wave and wave + 16 of the
// segment) stay in registers for the whole launch and a hundred kilobytes of requests are always out.  Eight waves
// with three blocks each left too little to cover a tile's LDS reads (34816 x 5120: 25.3 us, sixteen 23.2).  Cold, us,
// a tile per workgroup against the ring: 34816 x 5120 24.7 / 23.2, 43008 x 5120 29.4 / 26.9, 128256 x 4096 57.8 / 54.3,
// 57344 x 8192 61.1 / 48.3, 151936 x 5120 90.2 / 76.4 (5.7 TB/s).
// LDS map: [depth tiles of 16 x row_stride][a slot per wave; after the operands are read: row sums of 16 waves x 16, then
// the sums of all the workgroup's tiles].
template <int DT, int MAXB>
__device__ __forceinline__ void gemv_ring_body(const StreamParams& p) {
    constexpr uint32_t kBlock = StreamFormat<kQ4K>::kBytes;
    constexpr uint32_t kSlot = StreamFormat<kQ4K>::kSlot;
    constexpr uint32_t kAux = StreamFormat<kQ4K>::kAux;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t first = blockIdx.y * p.seg_blocks, nb = min(p.seg_blocks, p.nb - first);
    const uint32_t row_bytes = nb * kBlock, full_row_bytes = p.nb * kBlock;
    const uint32_t tiles = (p.n + 15u) / 16u;
    const uint32_t count = (tiles - blockIdx.x + gridDim.x - 1u) / gridDim.x;   // tiles blockIdx.x + i gridDim.x
    uint8_t* const slot = lds + p.depth * p.tile_bytes + wave * kSlot;
    float* const rsum = reinterpret_cast<float*>(lds + p.depth * p.tile_bytes);
    float* const sums = rsum + 256;

    // 1. the activations, as in the kernel above
    const size_t xrow = (size_t)first * 256u;
    typename std::conditional<DT == FH_F32, u32x4, u32x2>::type xraw[MAXB];
#pragma unroll
    for (int i = 0; i < MAXB; ++i) {
        const uint32_t b = min(wave + 16u * i, nb - 1u);
        if constexpr (DT == FH_F32) {
            const float* src = static_cast<const float*>(p.x) + xrow + b * 256u + lane * 4u;
            asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(xraw[i]) : "v"(src) : "memory");
        } else {
            const uint16_t* src = static_cast<const uint16_t*>(p.x) + xrow + b * 256u + lane * 4u;
            asm volatile("global_load_dwordx2 %0, %1, off" : "=v"(xraw[i]) : "v"(src) : "memory");
        }
    }
    // 2. a tile's requests: every wave asks for one row, a kilobyte per instruction; rows past the last repeat it, so that
    // every tile is the same number of instructions
    const uint32_t per_row = (row_bytes + 1023u) >> 10;
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
    auto request = [&](uint32_t it, uint32_t buffer) {
        const uint32_t row0 = (blockIdx.x + it * gridDim.x) * 16u;
        const uint8_t* const base = p.w + (size_t)min(row0 + wave, p.n - 1u) * full_row_bytes + first * kBlock;
        const uint32_t to = lds_base + buffer * p.tile_bytes + wave * p.row_stride;
        for (uint32_t c = 0; c < per_row; ++c)
            if (c * 1024u + lane * 16u < row_bytes) lds_load16_at(base, c * 1024u + lane * 16u, to + c * 1024u);
    };
    const uint32_t ahead = min(p.depth, count);
    for (uint32_t it = 0; it < ahead; ++it) request(it, it);
    if (lane < 4u) reinterpret_cast<uint32_t*>(slot + 1024u + kAux)[lane] = 0u;

    // 3. operands into registers, through the wave's slot
    const uint32_t n = lane & 15u, g = lane >> 4;
    const bool active = (n >> 2) == g;
    const uint8_t* const xlane = active ? slot + (g * 4u + (n & 3u)) * 16u : slot + 1024u + kAux;
    const uint32_t xstep = active ? 256u : 0u;
    wait_vmcnt(ahead * per_row);
    u32x4 xa[MAXB][4];
    float4 aux[MAXB];
#pragma unroll
    for (int i = 0; i < MAXB; ++i) {
        asm volatile("" : "+v"(xraw[i])::"memory");
        float4 v;
        if constexpr (DT == FH_F32) {
            v = make_float4(__uint_as_float(xraw[i].x), __uint_as_float(xraw[i].y), __uint_as_float(xraw[i].z),
                            __uint_as_float(xraw[i].w));
        } else if constexpr (DT == FH_F16) {
            v = make_float4(f16_bits_to_f32(xraw[i].x & 0xffffu), f16_bits_to_f32(xraw[i].x >> 16),
                            f16_bits_to_f32(xraw[i].y & 0xffffu), f16_bits_to_f32(xraw[i].y >> 16));
        } else {
            v = make_float4(bf16_bits_to_f32(xraw[i].x & 0xffffu), bf16_bits_to_f32(xraw[i].x >> 16),
                            bf16_bits_to_f32(xraw[i].y & 0xffffu), bf16_bits_to_f32(xraw[i].y >> 16));
        }
        stage_block(v, slot, lane);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // written before other lanes read it
#pragma unroll
        for (int u = 0; u < 4; ++u) xa[i][u] = *reinterpret_cast<const u32x4*>(xlane + u * xstep);
        aux[i] = *reinterpret_cast<const float4*>(slot + 1024u + 16u * g);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // read before the next block is written
    }

    // 4. the tiles in turn.  The barriers are bare: a __syncthreads would wait for the tiles on their way
    uint32_t buffer = 0;
    for (uint32_t it = 0; it < count; ++it) {
        wait_vmcnt(min(p.depth - 1u, count - 1u - it) * per_row);   // this tile has landed, the later ones may be out
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < MAXB; ++i) {
            const uint32_t b = wave + 16u * i;
            if (b < nb) {
                const uint8_t* const blk = lds + buffer * p.tile_bytes + n * p.row_stride + b * kBlock;
                const uint4 hdr = *reinterpret_cast<const uint4*>(blk);
                const uint4 qa = *reinterpret_cast<const uint4*>(blk + 16u + 32u * g);
                const uint4 qb = *reinterpret_cast<const uint4*>(blk + 32u + 32u * g);
                acc = multiply_q4k(xa[i], aux[i], hdr, qa, qb, g, acc);
            }
        }
        acc += __shfl_xor(acc, 16, 64);
        acc += __shfl_xor(acc, 32, 64);
        if (lane < 16u) rsum[wave * 16u + lane] = acc;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // every wave has read its part of the tile
        if (it + p.depth < count) request(it + p.depth, buffer);
        buffer = buffer + 1u == p.depth ? 0u : buffer + 1u;
        if (tid < 16u) {
            float total = 0.f;
#pragma unroll
            for (int w = 0; w < 16; ++w) total += rsum[w * 16 + tid];
            sums[it * 16u + tid] = total;
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the last tile's wait was for all there are)
    __syncthreads();

    // 5. out, or to the scratch: the last of a row group's segments adds all of them, in segment order
    auto row_of = [&](uint32_t i) { return (blockIdx.x + (i >> 4) * gridDim.x) * 16u + (i & 15u); };
    if (p.segments == 1) {
        for (uint32_t i = tid; i < count * 16u; i += 1024u)
            if (row_of(i) < p.n) store_from_f32(p.y, row_of(i), p.y_dtype, sums[i]);
        return;
    }
    for (uint32_t i = tid; i < count * 16u; i += 1024u)
        if (row_of(i) < p.n)
            __hip_atomic_store(&p.partials[(size_t)blockIdx.y * p.n + row_of(i)], sums[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the stores above have completed
    __syncthreads();
    uint32_t* const flag = reinterpret_cast<uint32_t*>(rsum);
    if (tid == 0) {
        uint32_t* counter = p.counters + blockIdx.x;
        const uint32_t ticket = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t last = ticket == p.segments - 1 ? 1u : 0u;
        if (last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *flag = last;
    }
    __syncthreads();
    if (*flag == 0) return;
    for (uint32_t i = tid; i < count * 16u; i += 1024u) {
        if (row_of(i) >= p.n) continue;
        float total = 0.f;
        for (uint32_t sg = 0; sg < p.segments; ++sg)
            total += __hip_atomic_load(&p.partials[(size_t)sg * p.n + row_of(i)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        store_from_f32(p.y, row_of(i), p.y_dtype, total);
    }
}

template <int DT, int MAXB>
__global__ __launch_bounds__(1024) void gemv_ring_q4k(const StreamParams p) {
    gemv_ring_body<DT, MAXB>(p);
}

}  // namespace

// The ring's plan: sixteen-row tiles of as few K segments as leave a wave two super-blocks and LDS room for two tiles.
static bool ring_plan(uint32_t n, uint32_t nb, uint32_t cus, StreamPlan* plan) {
    const uint32_t tiles = (n + 15u) / 16u, wanted = (nb + 23u) / 24u;
    const uint32_t seg = (nb + wanted - 1u) / wanted, segments = (nb + seg - 1u) / seg;
    const uint32_t stride = ((kQ4Bytes * seg) / 16u | 1u) * 16u, tile = 16u * stride, slots = 16u * kSlotBytes;
    const uint32_t per_row = (kQ4Bytes * seg + 1023u) / 1024u;
    uint32_t depth = (160u * 1024u - slots) / tile;
    if (depth > 4u) depth = 4u;
    if (depth * per_row > 20u) depth = 20u / per_row;   // the waits count to twenty
    const uint32_t most = cus / segments, groups = most < tiles ? most : tiles;
    // (the sums of a workgroup's tiles take the slots' room)
    if (depth < 2u || groups == 0 || ((tiles + groups - 1u) / groups) * 64u + 1024u > slots) return false;
    *plan = StreamPlan{true, 16u, groups, 16u, stride, depth * tile + slots, segments, seg, depth};
    return true;
}

// Tile height that spreads the rows evenly: the fewest 16-row rounds per compute unit, then the
// smallest height that still fits them.
StreamPlan gemv_stream_plan(uint32_t ggml_type, uint32_t n, uint32_t k, uint32_t m, int cu_count, bool any_size,
                            int forced_segments, int ring, bool f32_rows) {
    StreamPlan plan{};
    const bool q6 = ggml_type == kQ6K;
    const uint32_t block = q6 ? kQ6Bytes : kQ4Bytes, slot = q6 ? kSlot6Bytes : kSlotBytes;
    const uint32_t nb = k / 256u;
    const uint32_t cus = cu_count > 0 ? (uint32_t)cu_count : 256u;
    const uint32_t rounds = ((n + 15u) / 16u + cus - 1u) / cus;
    uint32_t h = (n + cus * rounds - 1u) / (cus * rounds);
    if (h > 16u) h = 16u;
    if (h < 1u) h = 1u;
    // A tile stays below 64 KB -- 69 KB for Q6_K, whose workgroups share a compute unit in twos and
    // whose sixteen rows of 5120 weights are 66 KB -- so that two or three workgroups share a compute
    // unit's LDS (the LDS-direct loads themselves reach every LDS address: M0 values of 69632, 135168
    // and 150000 were written to and read back on this device), and a wave owns at most six
    // super-blocks: longer rows are cut into K segments of equal length.
    const uint32_t tile_cap = q6 ? 80u * 1024u - 8u * slot - 8u * 64u : 65536u;
    auto stride_of = [block](uint32_t blocks) {
        uint32_t units = (block * blocks + 15u) / 16u;   // bytes / 16
        if ((units & 1u) == 0) ++units;    // odd number of 16-byte units: 16 rows start in 16 different bank groups
        return units * 16u;
    };
    // ... and, where it must be cut anyway, short enough that three workgroups share a compute
    // unit's LDS (the headline's uncut 14 x 2896 bytes do)
    const uint32_t budget = (160u * 1024u) / 3u - 8u * slot - 8u * 64u;
    // (the segments then spread the work, so the tiles are as tall as the matrix instruction)
    // the reference's K-split switch asks for at least that many segments, as far as whole blocks go
    const uint32_t wanted = forced_segments > 1 ? ((uint32_t)forced_segments < nb ? (uint32_t)forced_segments : nb) : 1u;
    if (wanted > 1u || nb > 48u || h * stride_of(nb) > tile_cap) h = n < 16u ? n : 16u;
    uint32_t segments = wanted, seg = (nb + wanted - 1u) / wanted;
    // LDS-direct loads want dword-aligned addresses: a Q6_K segment starts on an even block
    auto even_up = [q6](uint32_t blocks) { return q6 ? (blocks + 1u) & ~1u : blocks; };
    if (segments > 1u) seg = even_up(seg);
    while (seg > 48u || h * stride_of(seg) > (segments == 1 ? tile_cap : budget)) {
        ++segments;
        seg = even_up((nb + segments - 1u) / segments);
        if (seg <= (q6 ? 2u : 1u)) break;
    }
    segments = (nb + seg - 1u) / seg;
    plan.segments = segments;
    plan.seg_blocks = seg;
    plan.row_stride = stride_of(seg);
    if (h * plan.row_stride > tile_cap) h = tile_cap / plan.row_stride;
    plan.tile_rows = h;
    plan.tiles = (n + h - 1u) / h;
    plan.waves = 8u;
    plan.lds_bytes = h * plan.row_stride + plan.waves * slot + plan.waves * 64u;
    // Matrices of a megabyte or two finish sooner on the FMA kernel's smaller workgroups.  A Q6_K tile is 46% longer and
    // only two share a compute unit: rows that must be cut into segments in any case gain (5120 x 17408: 25.2 / 21.5), and so do large
    // matrices (us, weights out of every cache, FMA against this kernel: 34816 x 5120 36.5 / 32.7, 128256 x 4096 92 / 84, 152064 x 3584
    // 105 / 90, 151936 x 5120 137 / 117; profiles/waits_loads_lookups_us.txt).
    // Rows of 16 bits gain 1% there and are 0.9e-7 from 64 bits on the FMA kernel against 0.95e-7 here (f32 rows 1.9e-7 against
    // 0.9e-7), and two or three f32 rows share their weights through the caches on the FMA kernel (2 x 34816 x 5120 58.3 us there
    // against 64.6, 2 x 100000 x 2048 67.6 / 74.5): they come from a million super-blocks on, where the FMA kernel
    // cannot cut a row evenly over its eight block slots.
    // One f32 row of eight super-blocks and more gains from a quarter of a million of them on, whole or cut (22000 x 3072 16.3 / 15.0,
    // 17408 x 5120 21.9 / 20.1, 60000 x 2048 27.2 / 24.8, 36000 x 3584 29.8 / 26.5, 12000 x 10240 33.6 / 27.7; but 9000 x 6144 14.8 / 15.4,
    // 5120 x 8192 11.6 / 12.9, 7000 x 4096 7.8 / 8.3, and of shorter rows 40000 x 1536 16.8 / 16.1, 100000 x 1024 22.0 / 28.6).
    // Cut rows only while their partial sums fit any scratch, the fixed one of calls that must not allocate among them: the FMA kernel
    // would need none.
    const uint64_t blocks = (uint64_t)n * nb;
    const bool big_head = q6 && (f32_rows && m == 1 ? (nb >= 8u && blocks >= 250000u && (segments == 1u || (uint64_t)segments * n <= 100000u)) || (segments == 1u && h == 16u && blocks >= 600000u)
                                                    : segments == 1u && h == 16u && (nb & 7u) != 0 && blocks >= 1000000u);
    // One row of a Q4_K matrix of short rows is the FMA kernel's: a tile of sixteen is a few kilobytes of LDS for eight waves of
    // which some own no super-block, and staging stands beside little arithmetic (us, cold, FMA against this kernel:
    // 29952 x 256 3.7 / 8.3, 8448 x 512 3.5 / 4.2, 4224 x 1024 3.5 / 3.8, 99968 x 1024 14.1 / 23.6; rows of 5 - 8 super-blocks
    // 4992 x 1536 4.4 / 4.2, 12480 x 2048 5.8 / 6.0, 24960 x 1536 8.4 / 9.1, 156224 x 2048 40.7 / 48.3; of 9 - 12
    // 16640 x 3072 9.9 / 9.0, 40000 x 2560 16.0 / 16.0, 49984 x 2560 18.8 / 19.6, 104128 x 3072 34.6 / 38.8; of 14
    // 89280 x 3584 39.8 / 37.8).
    const uint64_t short_from = nb <= 4u ? 0u : nb <= 8u ? 100000u : nb <= 12u ? 450000u : ~0ull;
    const bool short_rows = m == 1 && (uint64_t)n * nb >= short_from;
    const bool wins = q6 ? nb > 48u || big_head : (uint64_t)n * nb >= 16384u && !short_rows;
    plan.ok = nb >= 1 && seg >= 1u && seg <= 48u && segments <= 65535u && h >= 1u && (any_size || wins) &&
              plan.lds_bytes <= 160u * 1024u && m >= 1 && m <= 65535u && (!q6 || (nb & 1u) == 0);
    if (!q6 && m == 1 && forced_segments <= 1 && ring != 0 && (any_size || plan.ok)) {
        // The ring pays its start, some 4 us without a tile finished, and the last round of tiles back on 100 MB of
        // weights in rows of 5120 and more (us, cold, a tile per workgroup against the ring: 34816 x 5120 24.7 / 23.2, 52032
        // x 6144 40.2 / 35.6, 39040 x 8192 43.6 / 37.2, 25984 x 12288 42.3 / 36.3, 18368 x 17408 42.4 / 38.6; but 22080 x 7168
        // 22.6 / 23.4, 17408 x 5120 12.9 / 15.5).  Shorter rows leave some of the sixteen waves idle: 69440 x 4608
        // 36.2 / 37.4, 89280 x 3584 37.8 / 37.7.
        const bool ring_wins = nb >= 20u && (uint64_t)n * nb >= 680000u;
        StreamPlan other{};
        if ((ring == 2 || ring_wins) && ring_plan(n, nb, cus, &other)) return other;
    }
    return plan;
}

const char* launch_gemv_stream(hipStream_t s, const GemvArgs& a, const StreamPlan& plan) {
    StreamParams p{};
    p.w = static_cast<const uint8_t*>(a.w);
    p.x = a.x;
    p.y = a.y;
    p.n = a.n;
    p.nb = a.k / 256u;
    p.tile_rows = plan.tile_rows;
    p.row_stride = plan.row_stride;
    p.tile_bytes = plan.tile_rows * plan.row_stride;
    p.x_dtype = a.x_dtype;
    p.y_dtype = a.y_dtype;
    p.segments = plan.segments;
    p.seg_blocks = plan.seg_blocks;
    p.m = a.m;
    p.partials = a.partials;
    p.counters = a.counters;
    p.depth = plan.depth;
    typedef void (*Kernel)(const StreamParams);
    // [format][dtype][blocks per wave: 2, 3, 6]
    static const Kernel kernels[2][3][3] = {
        {{gemv_stream_q4k<FH_F32, 8, 2>, gemv_stream_q4k<FH_F32, 8, 3>, gemv_stream_q4k<FH_F32, 8, 6>},
         {gemv_stream_q4k<FH_F16, 8, 2>, gemv_stream_q4k<FH_F16, 8, 3>, gemv_stream_q4k<FH_F16, 8, 6>},
         {gemv_stream_q4k<FH_BF16, 8, 2>, gemv_stream_q4k<FH_BF16, 8, 3>, gemv_stream_q4k<FH_BF16, 8, 6>}},
        {{gemv_stream_q6k<FH_F32, 8, 2>, gemv_stream_q6k<FH_F32, 8, 3>, gemv_stream_q6k<FH_F32, 8, 6>},
         {gemv_stream_q6k<FH_F16, 8, 2>, gemv_stream_q6k<FH_F16, 8, 3>, gemv_stream_q6k<FH_F16, 8, 6>},
         {gemv_stream_q6k<FH_BF16, 8, 2>, gemv_stream_q6k<FH_BF16, 8, 3>, gemv_stream_q6k<FH_BF16, 8, 6>}},
    };
    static std::atomic<uint64_t> raised{0};
    once_per_device(raised, [] {
        for (const auto& format : kernels)
            for (const auto& row : format)
                for (Kernel kernel : row)
                    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    });
    if (plan.depth != 0) {
        // [dtype][super-blocks per wave: 1, 2]
        static const Kernel rings[3][2] = {{gemv_ring_q4k<FH_F32, 1>, gemv_ring_q4k<FH_F32, 2>},
                                           {gemv_ring_q4k<FH_F16, 1>, gemv_ring_q4k<FH_F16, 2>},
                                           {gemv_ring_q4k<FH_BF16, 1>, gemv_ring_q4k<FH_BF16, 2>}};
        static std::atomic<uint64_t> ring_raised{0};
        once_per_device(ring_raised, [] {
            for (const auto& row : rings)
                for (Kernel kernel : row)
                    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        });
        p.tile_bytes = 16u * plan.row_stride;
        hipLaunchKernelGGL(rings[a.x_dtype][plan.seg_blocks > 16u ? 1 : 0], dim3(plan.tiles, plan.segments), dim3(16u * kWave),
                           plan.lds_bytes, s, p);
        return plan.segments > 1 ? "q4_k_gemv_ksplit" : "q4_k_gemv_factored";
    }
    const int shape = plan.seg_blocks <= 16u ? 0 : plan.seg_blocks <= 24u ? 1 : 2;
    const int format = a.ggml_type == kQ6K ? 1 : 0;
    // Q4_K tiles of up to 14 rows (two load instructions per super-block): every wave loads what it
    // multiplies and no workgroup barrier stands between the loads and the arithmetic.  Same box,
    // 17408 x 5120: 12.15 against 13.2 us and 12.3 against 12.4 us on two boxes (f16 activations 12.1
    // against 12.4); 5120 x 5120 6.5 either way.  Taller tiles need a third, nearly empty instruction
    // per block and lose (4096 x 4096: 4.54 against 4.40 us, 18992 x 5120: 14.0 against 13.8).
    const uint32_t own_bytes = plan.seg_blocks * plan.tile_rows * kQ4Bytes;
    if (a.stream_own && format == 0 && plan.tile_rows * (kQ4Bytes / 16u) <= 128u && own_bytes <= 65536u) {
        static const Kernel own_kernels[3][3] = {
            {gemv_stream_q4k_own<FH_F32, 8, 2>, gemv_stream_q4k_own<FH_F32, 8, 3>, gemv_stream_q4k_own<FH_F32, 8, 6>},
            {gemv_stream_q4k_own<FH_F16, 8, 2>, gemv_stream_q4k_own<FH_F16, 8, 3>, gemv_stream_q4k_own<FH_F16, 8, 6>},
            {gemv_stream_q4k_own<FH_BF16, 8, 2>, gemv_stream_q4k_own<FH_BF16, 8, 3>, gemv_stream_q4k_own<FH_BF16, 8, 6>},
        };
        Kernel kernel = own_kernels[a.x_dtype][shape];
        static std::atomic<uint64_t> own_raised{0};
        once_per_device(own_raised, [] {
            for (const auto& row : own_kernels)
                for (Kernel k : row)
                    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        });
        p.tile_bytes = own_bytes;
        const uint32_t lds = own_bytes + plan.waves * kSlotBytes + plan.waves * 64u;
        hipLaunchKernelGGL(kernel, dim3(plan.tiles, plan.segments, a.m), dim3(plan.waves * kWave), lds, s, p);
        return plan.segments > 1 ? "q4_k_gemv_ksplit" : "q4_k_gemv_factored";
    }
    hipLaunchKernelGGL(kernels[format][a.x_dtype][shape], dim3(plan.tiles, plan.segments, a.m), dim3(plan.waves * kWave),
                       plan.lds_bytes, s, p);
    if (format == 1) return plan.segments > 1 ? "q6_k_gemv_ksplit" : "q6_k_gemv_factored";
    return plan.segments > 1 ? "q4_k_gemv_ksplit" : "q4_k_gemv_factored";
}

}  // namespace fh
