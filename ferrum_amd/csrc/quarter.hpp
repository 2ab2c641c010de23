// The register decode shared by the kernels that stream weights past resident activation rows
// (gemm_skinny.hip, gemm_rows.hip).  Sixty-four lanes are 16 weight rows x 4 lane groups; a lane
// group owns one quarter of every super-block of its row (Q4_K: one 64-weight chunk, 32 contiguous
// bytes; Q6_K: 16 positions of one 128-weight half) and turns it into matrix operands in registers.
#pragma once

#include "device_utils.hpp"
#include "internal.hpp"
#include "tile_decode.hpp"

namespace fh {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // a native vector: copies stay in registers

// Operands for the 16-bit matrix instructions: every weight rounded once to the tile type.
template <int DT>
struct PackedOperands {
    uint32_t words[32];
    __device__ __forceinline__ void pair(int i, float qa, float qb, float scale, float offset) {
        words[i] = fma_pair<DT>(qa, qb, scale, offset);
    }
    __device__ __forceinline__ uint4 operand(int s) const {
        return make_uint4(words[4 * s], words[4 * s + 1], words[4 * s + 2], words[4 * s + 3]);
    }
};

// The exact f32 weights, for the f32 matrix instruction.
struct FloatOperands {
    float v[64];
    __device__ __forceinline__ void pair(int i, float qa, float qb, float scale, float offset) {
        v[2 * i] = fmaf(qa, scale, offset);
        v[2 * i + 1] = fmaf(qb, scale, offset);
    }
};

// One lane's quarter of a super-block, raw, and its decode into 8 matrix operands of 8 weights
// each: out.pair(i, qa, qb, scale, offset) receives weights 2i and 2i + 1 of the quarter in operand
// order as the two fmas q * scale + offset that give the exact f32 weight.
// klocal(g, s): K offset inside the super-block of the 8 weights of operand s.
template <uint32_t TYPE>
struct Quarter;

template <>
struct Quarter<kQ4K> {
    static constexpr uint32_t kBlockBytes = 144;
    static constexpr int kLoads = 3;   // memory instructions of load()
    uint4 hdr, qa, qb;
    __device__ __forceinline__ void load(const uint8_t* block, uint32_t g) {
        hdr = *reinterpret_cast<const uint4*>(block);
        qa = *reinterpret_cast<const uint4*>(block + 16 + 32 * g);
        qb = *reinterpret_cast<const uint4*>(block + 32 + 32 * g);
    }
    // operands 0..3: low nibbles (weights 64g + 8s ..), 4..7: high nibbles (64g + 32 + 8(s-4) ..)
    static __device__ __forceinline__ uint32_t klocal(uint32_t g, int s) { return 64 * g + 8 * s; }
    template <class Sink>
    __device__ __forceinline__ void decode_into(uint32_t g, Sink& out) const {
        const float d = f16_bits_to_f32(hdr.x & 0xffffu), dmin = f16_bits_to_f32(hdr.x >> 16);
        float sc0, sc1, mn0, mn1;
        q4k_chunk_scales(hdr.y, hdr.z, hdr.w, g, sc0, sc1, mn0, mn1);
        // d*sc and dmin*m are exact in f32; the powers of two undo the subnormal encoding
        const float a_lo = (d * sc0) * 16777216.f, a_hi = (d * sc1) * 1048576.f;
        const float b_lo = -(dmin * mn0), b_hi = -(dmin * mn1);
        const uint32_t v[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const uint32_t w0 = v[t], w1 = w0 >> 8;
            const uint32_t l02 = w0 & 0x000f000fu, h02 = w0 & 0x00f000f0u;
            const uint32_t l13 = w1 & 0x000f000fu, h13 = w1 & 0x00f000f0u;
            out.pair(2 * t, lo_half(l02), lo_half(l13), a_lo, b_lo);
            out.pair(2 * t + 1, hi_half(l02), hi_half(l13), a_lo, b_lo);
            out.pair(16 + 2 * t, lo_half(h02), lo_half(h13), a_hi, b_hi);
            out.pair(16 + 2 * t + 1, hi_half(h02), hi_half(h13), a_hi, b_hi);
        }
    }
};

template <>
struct Quarter<kQ5K> {
    static constexpr uint32_t kBlockBytes = 176;
    static constexpr int kLoads = 5;   // memory instructions of load()
    uint4 hdr, ha, hb, qa, qb;   // ha, hb: the block's 32 qh bytes (fifth bits, bit 2g low / 2g + 1 high nibbles)
    __device__ __forceinline__ void load(const uint8_t* block, uint32_t g) {
        hdr = *reinterpret_cast<const uint4*>(block);
        ha = *reinterpret_cast<const uint4*>(block + 16);
        hb = *reinterpret_cast<const uint4*>(block + 32);
        qa = *reinterpret_cast<const uint4*>(block + 48 + 32 * g);
        qb = *reinterpret_cast<const uint4*>(block + 64 + 32 * g);
    }
    static __device__ __forceinline__ uint32_t klocal(uint32_t g, int s) { return 64 * g + 8 * s; }
    template <class Sink>
    __device__ __forceinline__ void decode_into(uint32_t g, Sink& out) const {
        const float d = f16_bits_to_f32(hdr.x & 0xffffu), dmin = f16_bits_to_f32(hdr.x >> 16);
        float sc0, sc1, mn0, mn1;
        q4k_chunk_scales(hdr.y, hdr.z, hdr.w, g, sc0, sc1, mn0, mn1);
        const float a_lo = (d * sc0) * 16777216.f, a_hi = (d * sc1) * 1048576.f;
        const float b_lo = -(dmin * mn0), b_hi = -(dmin * mn1);
        const uint32_t v[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
        const uint32_t p[8] = {ha.x, ha.y, ha.z, ha.w, hb.x, hb.y, hb.z, hb.w};
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const uint32_t w0 = v[t], w1 = w0 >> 8;
            const uint32_t p0 = p[t] >> (2 * g), p1 = p0 >> 8;
            const uint32_t l02 = (w0 & 0x000f000fu) | ((p0 & 0x00010001u) << 4);
            const uint32_t l13 = (w1 & 0x000f000fu) | ((p1 & 0x00010001u) << 4);
            const uint32_t h02 = (w0 & 0x00f000f0u) | ((p0 & 0x00020002u) << 7);
            const uint32_t h13 = (w1 & 0x00f000f0u) | ((p1 & 0x00020002u) << 7);
            out.pair(2 * t, lo_half(l02), lo_half(l13), a_lo, b_lo);
            out.pair(2 * t + 1, hi_half(l02), hi_half(l13), a_lo, b_lo);
            out.pair(16 + 2 * t, lo_half(h02), lo_half(h13), a_hi, b_hi);
            out.pair(16 + 2 * t + 1, hi_half(h02), hi_half(h13), a_hi, b_hi);
        }
    }
};

// IQ4_XS: lane group g owns sub-blocks 2g and 2g + 1 (qs bytes [32g, +32)).  Low
// nibbles are a sub-block's weights 0..15, high nibbles 16..31, so operand s
// covers weights 64g + 8s .. as for Q4_K.  Codebook bytes (value + 128) become
// f16 subnormals; fma(byte, scale, -128 scale) is the exact weight.
template <>
struct Quarter<kIQ4XS> {
    static constexpr uint32_t kBlockBytes = 136;
    static constexpr int kLoads = 3;   // memory instructions of load()
    uint2 hdr;
    uint4 qa, qb;
    __device__ __forceinline__ void load(const uint8_t* block, uint32_t g) {
        hdr = *reinterpret_cast<const uint2*>(block);
        qa = load_u4_unaligned(block + 8 + 32 * g);
        qb = load_u4_unaligned(block + 24 + 32 * g);
    }
    static __device__ __forceinline__ uint32_t klocal(uint32_t g, int s) { return 64 * g + 8 * s; }
    template <class Sink>
    __device__ __forceinline__ void decode_into(uint32_t g, Sink& out) const {
        const uint32_t v[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            const float dl = iq4xs_scale(hdr.x, hdr.y, 2 * g + sub);
            const float scale = dl * 16777216.f, offset = -128.f * dl;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint32_t l = iq4_lookup4(v[4 * sub + t]), h = iq4_lookup4(v[4 * sub + t] >> 4);
                const uint32_t l02 = bytes02_as_halves(l), l13 = bytes13_as_halves(l);
                const uint32_t h02 = bytes02_as_halves(h), h13 = bytes13_as_halves(h);
                // weights 0..15 of the sub-block are its low nibbles, 16..31 its high ones
                out.pair(16 * sub + 2 * t, lo_half(l02), lo_half(l13), scale, offset);
                out.pair(16 * sub + 2 * t + 1, hi_half(l02), hi_half(l13), scale, offset);
                out.pair(16 * sub + 8 + 2 * t, lo_half(h02), lo_half(h13), scale, offset);
                out.pair(16 * sub + 8 + 2 * t + 1, hi_half(h02), hi_half(h13), scale, offset);
            }
        }
    }
};

// Q8_0: lane group g owns blocks 2g and 2g + 1 of the 256-weight run; operand s covers
// weights 64g + 8s .., two quant dwords of one block.
template <>
struct Quarter<kQ8_0> {
    static constexpr uint32_t kBlockBytes = 272;
    static constexpr int kLoads = 5;   // memory instructions of load()
    Q8Pair p;
    __device__ __forceinline__ void load(const uint8_t* block, uint32_t g) { p.load(block + 68 * g); }
    static __device__ __forceinline__ uint32_t klocal(uint32_t g, int s) { return 64 * g + 8 * s; }
    template <class Sink>
    __device__ __forceinline__ void decode_into(uint32_t, Sink& out) const {
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) {
            const float d = p.d(blk);
            const float scale = d * 16777216.f, offset = -128.f * d;   // fma(q + 128, d, -128 d) = d q, exact
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const uint32_t u0 = p.biased(blk, 2 * s), u1 = p.biased(blk, 2 * s + 1);
                const uint32_t a02 = bytes02_as_halves(u0), a13 = bytes13_as_halves(u0);
                const uint32_t b02 = bytes02_as_halves(u1), b13 = bytes13_as_halves(u1);
                const int word = 16 * blk + 4 * s;
                out.pair(word, lo_half(a02), lo_half(a13), scale, offset);
                out.pair(word + 1, hi_half(a02), hi_half(a13), scale, offset);
                out.pair(word + 2, lo_half(b02), lo_half(b13), scale, offset);
                out.pair(word + 3, hi_half(b02), hi_half(b13), scale, offset);
            }
        }
    }
};

template <>
struct Quarter<kQ6K> {
    static constexpr uint32_t kBlockBytes = 210;
    static constexpr int kLoads = 5;   // memory instructions of load()
    uint4 la, lb, ph, sc;
    uint32_t d;
    // lane group g: half h = g / 2 of the block, positions j0 = 16 (g & 1) .. j0 + 15
    __device__ __forceinline__ void load(const uint8_t* block, uint32_t g) {
        const uint32_t h = g >> 1, j0 = (g & 1u) * 16;
        la = load_u4_unaligned(block + 64 * h + j0);
        lb = load_u4_unaligned(block + 64 * h + 32 + j0);
        ph = load_u4_unaligned(block + 128 + 32 * h + j0);
        sc = load_u4_unaligned(block + 192);
        d = load_u16_unaligned(block + 208);
    }
    // out of LDS, `behind`: the block begins two bytes behind a dword, else at one
    __device__ __forceinline__ void load_by_dwords(const uint8_t* block, uint32_t g, bool behind) {
        const uint32_t h = g >> 1, j0 = (g & 1u) * 16;
        auto read = [behind](const uint8_t* p) { return behind ? lds_u4_behind_2(p) : lds_u4_dword(p); };
        la = read(block + 64 * h + j0);
        lb = read(block + 64 * h + 32 + j0);
        ph = read(block + 128 + 32 * h + j0);
        sc = read(block + 192);
        d = load_u16_unaligned(block + 208);
    }
    // operand s: slice s / 2 (32 weights each), positions j0 + 8 (s & 1) ..
    static __device__ __forceinline__ uint32_t klocal(uint32_t g, int s) {
        return 128 * (g >> 1) + 32 * (s >> 1) + 16 * (g & 1u) + 8 * (s & 1);
    }
    template <class Sink>
    __device__ __forceinline__ void decode_into(uint32_t g, Sink& out) const {
        const float df = f16_bits_to_f32(d);
        const uint32_t h = g >> 1;
        const uint32_t scw[4] = {sc.x, sc.y, sc.z, sc.w};
        const uint32_t lav[4] = {la.x, la.y, la.z, la.w}, lbv[4] = {lb.x, lb.y, lb.z, lb.w};
        const uint32_t phv[4] = {ph.x, ph.y, ph.z, ph.w};
        // scales 8h + 2*slice + (g & 1): slices 0,1 in word 2h, slices 2,3 in word 2h + 1
        const uint32_t w_lo = (h ? scw[2] : scw[0]) >> (8 * (g & 1u));
        const uint32_t w_hi = (h ? scw[3] : scw[1]) >> (8 * (g & 1u));
#pragma unroll
        for (int slice = 0; slice < 4; ++slice) {
            const uint32_t word = slice < 2 ? w_lo : w_hi;
            const float s = df * (float)(int)(int8_t)(word >> (16 * (slice & 1)));
            const float scale = s * ((slice < 2) ? 16777216.f : 1048576.f);  // high nibbles sit 4 bits up
            const float offset = -32.f * s;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint32_t w0 = (slice & 1) ? lbv[t] : lav[t], w1 = w0 >> 8;
                const uint32_t p0 = phv[t] >> (2 * slice), p1 = p0 >> 8;
                uint32_t q02, q13;
                if (slice < 2) {  // low nibble | plane bits << 4 : q * 2^-24
                    q02 = (w0 & 0x000f000fu) | ((p0 & 0x00030003u) << 4);
                    q13 = (w1 & 0x000f000fu) | ((p1 & 0x00030003u) << 4);
                } else {          // high nibble in place | plane bits << 8 : 16 q * 2^-24
                    q02 = (w0 & 0x00f000f0u) | ((p0 & 0x00030003u) << 8);
                    q13 = (w1 & 0x00f000f0u) | ((p1 & 0x00030003u) << 8);
                }
                out.pair(8 * slice + 2 * t, lo_half(q02), lo_half(q13), scale, offset);
                out.pair(8 * slice + 2 * t + 1, hi_half(q02), hi_half(q13), scale, offset);
            }
        }
    }
};

}  // namespace fh
