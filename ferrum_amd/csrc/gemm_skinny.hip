// Routed-expert projections (f16 / bf16 activations grouped by expert) on the matrix cores,
// Y = X . W[expert]^T for Q4_K / Q5_K / Q6_K / IQ4_XS / Q8_0 weights, and the dense product whose
// rows stay in LDS.
//
// With an expert's few tokens the job is a weight stream (HBM bound), so nothing of
// the weights goes through LDS.  A wave owns 16 weight rows.  Its 64 lanes are
// 16 rows x 4 lane groups, and a lane group owns one quarter of every
// super-block of its row (Q4_K: one 64-weight chunk, 32 contiguous bytes;
// Q6_K: 16 positions of one 128-weight half).  The lane decodes its 64 weights
// in registers straight into eight A operands of v_mfma_f32_16x16x32 (rows =
// weight rows): an MFMA only needs A and B to agree on which 32 K indices a
// step covers, so step s simply takes "the s-th run of 8 weights of every lane
// group's quarter", and the activations are read from LDS in the same order.
// Decoding is the one-rounding fma of tile_decode.hpp, so tile values carry the
// bits of the reference's dequantisation rounded once to the tile type.
//
// gemm_skinny_kernel, for rows too wide for LDS: the four waves of a workgroup cover 64 rows and share the activation slab
// (16*TT tokens x 256 K) of the current super-block through a double-buffered
// LDS tile; one barrier per super-block.  Every lane keeps kRing super-blocks
// and kRing activation slabs in flight in registers: loads return in order, so
// both rings must run equally far ahead or the nearer one would drain the
// farther.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "device_utils.hpp"
#include "lds_direct.hpp"
#include "quarter.hpp"
#include "tile_decode.hpp"
#include "internal.hpp"

namespace fh {
namespace {

constexpr int kSkThreads = 256;
constexpr int kSkRows = 64;         // weight rows per workgroup
constexpr int kSlabLd = 256 + 8;    // halfs per token row of the LDS slab (16-byte skew)
constexpr int kRing = 5;

// One thread's share of an activation slab (16*TT tokens x 256 K) on its way
// from global memory to LDS.

template <int XP>
struct SlabRows {
    const uint16_t* row[XP];  // activation row of the token each piece belongs to, at this thread's column
};

template <int XP>
struct SlabRegs {
    u32x4 v[XP];
    __device__ __forceinline__ void load(const SlabRows<XP>& rows, size_t col) {
#pragma unroll
        for (int p = 0; p < XP; ++p) v[p] = *reinterpret_cast<const u32x4*>(rows.row[p] + col);
    }
    __device__ __forceinline__ void store(uint16_t* dst) const {
#pragma unroll
        for (int p = 0; p < XP; ++p) *reinterpret_cast<u32x4*>(dst + p * 8 * kSlabLd) = v[p];
    }
};

// blockIdx.y is an expert; its
// tokens are the assignments order[offsets[e]] .. order[offsets[e+1] - 1], or rows
// offsets[e] .. offsets[e+1] - 1 themselves when order is null (rows
// of x and of y), its weights rows [e*n, e*n + n), and the workgroup makes as
// many passes of 16*TT tokens as the expert's count needs (the weights of the
// later passes come from L2).
template <uint32_t TYPE, int DT, int TT>
__global__ __launch_bounds__(kSkThreads) void gemm_skinny_kernel(const uint8_t* __restrict__ w,
                                                                 const uint16_t* __restrict__ x,
                                                                 void* __restrict__ y, uint32_t m,
                                                                 uint32_t n, uint32_t nb,
                                                                 uint32_t y_dtype,
                                                                 const uint32_t* __restrict__ offsets,
                                                                 const uint32_t* __restrict__ order) {
    constexpr uint32_t kBB = Quarter<TYPE>::kBlockBytes;
    constexpr int kTokens = 16 * TT;
    constexpr int kSlab = kTokens * kSlabLd;      // halfs per LDS buffer
    constexpr int kXP = 2 * TT;                   // 16-byte pieces of a slab per thread
    __shared__ __attribute__((aligned(16))) uint16_t slab[2 * kSlab];

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t r = lane & 15u, g = lane >> 4;
    const uint32_t row0 = blockIdx.x * kSkRows + wave * 16;
    const uint32_t row = min(row0 + r, n - 1);
    const size_t k = (size_t)nb * 256;

    // a damaged offsets table reads wrong rows, never rows outside the m assignments
    const uint32_t first_token = min(offsets[blockIdx.y], m);
    const uint32_t upto = min(offsets[blockIdx.y + 1], m);
    const uint32_t count = upto > first_token ? upto - first_token : 0;
    const size_t expert_row = (size_t)blockIdx.y * n;
    const uint8_t* wrow = w + (expert_row + row) * nb * kBB;

    // activation slab pieces of this thread: piece p covers token 8p + tid / 32, halfs
    // 8 (tid % 32) ..
    const uint32_t xtok = tid >> 5, xcol = 8 * (tid & 31u);
    const uint32_t xdst = xtok * kSlabLd + xcol;

    // B operand address of (token r of tile tt, step s) inside a slab
    uint32_t boff[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) boff[s] = r * kSlabLd + Quarter<TYPE>::klocal(g, s);
    const uint32_t last = nb - 1;

    for (uint32_t t0 = 0; t0 < count; t0 += kTokens) {
        const uint32_t mt = min((uint32_t)kTokens, count - t0);
        if (t0 != 0) __syncthreads();  // the previous pass is done with the slabs
        // tokens past the count repeat the last one (their output columns are never
        // stored), which keeps the loop free of branches
        SlabRows<kXP> rows;
#pragma unroll
        for (int p = 0; p < kXP; ++p) {
            uint32_t token = first_token + t0 + min(xtok + 8 * p, mt - 1);
            token = order != nullptr ? order[token] : token;
            rows.row[p] = x + (size_t)token * k + xcol;
        }

        SlabRegs<kXP> xr[kRing];
        Quarter<TYPE> ring[kRing];
        // ring[i] holds super-block j with j % kRing == i; xr[i] holds activation slab j + 1
        {
            SlabRegs<kXP> first;
            first.load(rows, 0);
#pragma unroll
            for (int i = 0; i < kRing; ++i) {
                ring[i].load(wrow + (size_t)min((uint32_t)i, last) * kBB, g);
                xr[i].load(rows, 256 * (size_t)min((uint32_t)i + 1, last));
                // issue order matters: the loop waits by count, oldest first
                __builtin_amdgcn_sched_barrier(0);
            }
            first.store(slab + xdst);
        }

        float4v acc[TT];
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[t] = float4v{0.f, 0.f, 0.f, 0.f};

        auto multiply = [&](const PackedOperands<DT>& a, uint32_t buf) {
            const uint16_t* sl = slab + buf * kSlab;
#pragma unroll
            for (int s = 0; s < 8; ++s) {
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    const uint4 bfrag = *reinterpret_cast<const uint4*>(sl + boff[s] + t * 16 * kSlabLd);
                    acc[t] = mfma16<DT>(a.operand(s), bfrag, acc[t]);
                }
            }
        };

        uint32_t b = 0;
        // Full rings, straight-line: a load that would run past the row re-reads the
        // last super-block / slab instead (a cache hit that is never used), so the
        // loop body has no branch and the outstanding-load counts stay exact.
        for (; b + kRing <= nb; b += kRing) {
#pragma unroll
            for (int i = 0; i < kRing; ++i) {
                const uint32_t j = b + i;
                __syncthreads();
                // keep the scheduler from pulling a later super-block's decode up to here:
                // it would have to wait for that block's loads and drain the ring
                __builtin_amdgcn_sched_barrier(0);
                xr[i].store(slab + ((j + 1) & 1u) * kSlab + xdst);
                xr[i].load(rows, 256 * (size_t)min(j + 1 + kRing, last));
                PackedOperands<DT> a;
                ring[i].decode_into(g, a);
                ring[i].load(wrow + (size_t)min(j + kRing, last) * kBB, g);
                multiply(a, j & 1u);
            }
        }
        // the nb % kRing super-blocks left over are already in registers
#pragma unroll
        for (int i = 0; i < kRing - 1; ++i) {
            const uint32_t j = b + i;
            if (j < nb) {
                __syncthreads();
                xr[i].store(slab + ((j + 1) & 1u) * kSlab + xdst);
                PackedOperands<DT> a;
                ring[i].decode_into(g, a);
                multiply(a, j & 1u);
            }
        }

        // C layout of 16x16x32: acc[t][v] = (weight row 4g + v, token 16t + r)
        const uint32_t out_row = row0 + 4 * g;
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const uint32_t tok = 16 * t + r;
            if (tok >= mt) continue;
            uint32_t token = first_token + t0 + tok;
            token = order != nullptr ? order[token] : token;
            const size_t base = (size_t)token * n + out_row;
            if (y_dtype == FH_F32 && (n & 3u) == 0 && out_row + 3 < n) {
                *reinterpret_cast<float4*>(static_cast<float*>(y) + base) =
                    make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (out_row + v < n) store_from_f32(y, base + v, y_dtype, acc[t][v]);
            }
        }
    }
}

// Routed-expert projection with the expert's activations resident in LDS.
// When an expert's tokens (16*TT of them at a time) fit LDS for the whole K, a
// workgroup gathers them once and then streams weight rows past them with no
// further barrier: wave w takes row tiles w, w+4, ... of the workgroup's share
// and walks (tile, super-block) units through a register ring, so the prefetch
// runs across tile boundaries.  blockIdx.y = expert, blockIdx.x = which share
// of the expert's rows.  Dynamic LDS: 16*TT rows of K halfs.
//
// The rows are [A, K] rows or, with metadata given, the row of the assignment's
// token in [tokens, K]: expert_assign folded into the gather.  (SiLU * up is not
// folded in: it is bound by its exponentials and divisions, and one workgroup
// per compute unit doing them ahead of its first MFMA costs more than the
// launch that spreads them over the whole chip: +11 us against -5 us.)
constexpr size_t kResLdsBytes = 160u * 1024;   // a workgroup may take all of a compute unit's LDS
constexpr int kResRing = 6;
constexpr int kResWaves = 8;                    // two waves per SIMD hide each other's decode and MFMA waits
constexpr int kResThreads = 64 * kResWaves;

// A shared expert in the same launch: every token also runs the dense matrix w [n, k];
// token t reads row t of x (null: row t of the routed x, which then holds token rows) and
// writes row t of y.  Its work is cut into pieces of 16*TT consecutive tokens times
// tiles_per_slice row tiles, `slices` of them per token group, and the workgroups share the
// pieces out after their own expert, so the grid and its one round of workgroups stay as
// they are.
struct ResidentShared {
    const uint8_t* w;
    const uint16_t* x;
    void* y;
    uint32_t tokens;
    uint32_t slices;
    uint32_t tiles_per_slice;
};

// Copies `mt` activation rows into LDS for the resident kernels: row `tok` of the item to
// xs[tok * ld ..], its 16-byte pieces swizzled by the row's low four bits; eight pieces per thread
// in flight at a time.  The row behind a slot is found through up to two tables (the expert-sorted
// order, then the assignment's token).  All eight pieces look their rows up together, table by
// table, before any row is read: a round trip per table and one for the rows, where piece after
// piece would chain up to twenty-four.  F32: the rows are f32 and rounded to f16 on the way, as
// launch_round_to_f16 rounds them: a launch for the routed rows, one for the shared expert's and a
// trip through memory less per projection (1600 routes of 200 tokens, 256 IQ4_XS experts: 116 us for
// the three launches of a 1024 x 2048 projection, 70 of a 2048 x 512 one; 104 and 58 for one).
template <bool F32>
__device__ __forceinline__ void gather_rows(uint16_t* xs, const uint16_t* __restrict__ xsrc, uint32_t mt,
                                            uint32_t pieces, uint32_t k, uint32_t ld, uint32_t first_token,
                                            const uint32_t* __restrict__ order, const float* __restrict__ metadata,
                                            uint32_t x_rows, uint32_t tid) {
    const uint32_t total = mt * pieces;
    for (uint32_t base = 0; base < total; base += 8 * kResThreads) {
        u32x4 v[8];
        uint32_t dst[8], row[8], pc[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t idx = min(base + j * kResThreads + tid, total - 1);
            const uint32_t tok = idx / pieces;
            pc[j] = idx - tok * pieces;
            dst[j] = tok * ld + 8 * (pc[j] ^ (tok & 15u));
            row[j] = first_token + tok;  // without tables a slot is its row
        }
        if (order != nullptr) {
#pragma unroll
            for (int j = 0; j < 8; ++j) row[j] = order[row[j]];
        }
        if (metadata != nullptr) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint32_t token = __float_as_uint(metadata[3 * (size_t)row[j] + 1]);
                row[j] = token < x_rows ? token : x_rows - 1;
            }
        }
        if constexpr (F32) {
            const float* const source = reinterpret_cast<const float*>(xsrc);
            float4 lo[8], hi[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float4* const at = reinterpret_cast<const float4*>(source + (size_t)row[j] * k + 8 * (size_t)pc[j]);
                lo[j] = at[0];
                hi[j] = at[1];
            }
#pragma unroll
            for (int j = 0; j < 8; ++j)
                v[j] = u32x4{f32_to_f16_bits(lo[j].x) | (f32_to_f16_bits(lo[j].y) << 16),
                             f32_to_f16_bits(lo[j].z) | (f32_to_f16_bits(lo[j].w) << 16),
                             f32_to_f16_bits(hi[j].x) | (f32_to_f16_bits(hi[j].y) << 16),
                             f32_to_f16_bits(hi[j].z) | (f32_to_f16_bits(hi[j].w) << 16)};
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                v[j] = *reinterpret_cast<const u32x4*>(xsrc + (size_t)row[j] * k + 8 * (size_t)pc[j]);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) *reinterpret_cast<u32x4*>(xs + dst[j]) = v[j];
    }
}

template <uint32_t TYPE, int DT, int TT, bool F32 = false>
__global__ __launch_bounds__(kResThreads) void expert_resident_kernel(const uint8_t* __restrict__ w,
                                                                     const uint16_t* __restrict__ x,
                                                                     void* __restrict__ y, uint32_t n,
                                                                     uint32_t nb, uint32_t y_dtype,
                                                                     const uint32_t* __restrict__ offsets,
                                                                     const uint32_t* __restrict__ order,
                                                                     uint32_t tiles_per_wg,
                                                                     const float* __restrict__ metadata,
                                                                     uint32_t x_rows, uint32_t routes,
                                                                     const ResidentShared sh) {
    constexpr uint32_t kBB = Quarter<TYPE>::kBlockBytes;
    constexpr int kTokens = 16 * TT;
    extern __shared__ __attribute__((aligned(16))) uint16_t xs[];

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t r = lane & 15u, g = lane >> 4;
    // Rows are not padded: 16 rows of 5120 halves are all of LDS.  The 16-byte piece p of row t
    // sits at piece p ^ (t & 15) instead, so the sixteen rows a B-operand read touches at one k
    // (and the sixteen consecutive pieces a gather write covers) fall on different banks.
    const uint32_t k = nb * 256, ld = k;
    // no offsets: a dense product, all of it shared-expert pieces
    // a damaged offsets table reads wrong rows, never rows outside the `routes` assignments
    const uint32_t expert_first = offsets != nullptr ? min(offsets[blockIdx.y], routes) : 0;
    const uint32_t expert_upto = offsets != nullptr ? min(offsets[blockIdx.y + 1], routes) : 0;
    const uint32_t count = expert_upto > expert_first ? expert_upto - expert_first : 0;
    const uint32_t tiles = (n + 15) / 16;
    const uint32_t pieces = k / 8;  // 16-byte pieces per activation row

    // work items of this workgroup: its expert's tokens, 16*TT at a time, then its part of
    // the shared expert's pieces
    const uint32_t passes = (count + kTokens - 1) / kTokens;
    const uint32_t wg = blockIdx.y * gridDim.x + blockIdx.x, wgs = gridDim.x * gridDim.y;
    const uint32_t shared_pieces = sh.w != nullptr ? (sh.tokens + kTokens - 1) / kTokens * sh.slices : 0;
    const uint32_t my_pieces = shared_pieces > wg ? (shared_pieces - wg + wgs - 1) / wgs : 0;
    for (uint32_t item = 0; item < passes + my_pieces; ++item) {
        const bool shared = item >= passes;  // uniform over the workgroup
        uint32_t first_token, mt, tile_begin, tile_end;
        if (!shared) {
            first_token = expert_first + item * kTokens;
            mt = min((uint32_t)kTokens, count - item * kTokens);
            tile_begin = blockIdx.x * tiles_per_wg + wave;
            tile_end = min(tiles, (blockIdx.x + 1) * tiles_per_wg);
        } else {
            const uint32_t piece = wg + (item - passes) * wgs;
            const uint32_t group = piece / sh.slices, slice = piece - group * sh.slices;
            first_token = group * kTokens;
            mt = min((uint32_t)kTokens, sh.tokens - first_token);
            tile_begin = slice * sh.tiles_per_slice + wave;
            tile_end = min(tiles, (slice + 1) * sh.tiles_per_slice);
        }
        const uint8_t* wexpert = shared ? sh.w : w + (size_t)blockIdx.y * n * nb * kBB;
        const uint16_t* xsrc = shared && sh.x != nullptr ? sh.x : x;
        void* ydst = shared ? sh.y : y;
        if (item != 0) __syncthreads();  // the previous item is done with the rows
        gather_rows<F32>(xs, xsrc, mt, pieces, k, ld, first_token, shared ? nullptr : order, shared ? nullptr : metadata,
                    x_rows, tid);
        __syncthreads();
        if (tile_begin >= tile_end) continue;  // uniform per wave; no barrier follows in this item

        // B operand rows: token 16t + r, clamped (columns past mt are never stored)
        uint32_t boff[TT];
        uint32_t out_token[TT];
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const uint32_t tok = min(16u * t + r, mt - 1);
            boff[t] = tok * ld;
            out_token[t] = order != nullptr && !shared ? order[first_token + tok] : first_token + tok;
        }
        uint32_t kl[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) kl[s] = (((Quarter<TYPE>::klocal(g, s) >> 3) ^ r) << 3);  // row 16t + r: swizzle r

        // units = (tile, super-block) pairs of this wave, in order
        const uint32_t my_tiles = (tile_end - tile_begin + kResWaves - 1) / kResWaves;
        const uint32_t units = my_tiles * nb;
        auto unit_ptr = [&](uint32_t tile, uint32_t b) {
            const uint32_t row = min(tile * 16 + r, n - 1);
            return wexpert + ((size_t)row * nb + b) * kBB;
        };
        Quarter<TYPE> ring[kResRing];
        uint32_t ptile = tile_begin, pb = 0;  // next unit to prefetch
        auto prefetch = [&](Quarter<TYPE>& slot) {
            slot.load(unit_ptr(min(ptile, tile_end - 1), pb), g);
            if (++pb == nb) {
                pb = 0;
                ptile += kResWaves;
            }
        };
#pragma unroll
        for (int i = 0; i < kResRing; ++i) {
            prefetch(ring[i]);
            __builtin_amdgcn_sched_barrier(0);
        }

        float4v acc[TT];
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[t] = float4v{0.f, 0.f, 0.f, 0.f};
        uint32_t tile = tile_begin, b = 0;
        auto consume = [&](Quarter<TYPE>& slot) {
            PackedOperands<DT> a;
            slot.decode_into(g, a);
            prefetch(slot);
            const uint16_t* xb = xs + 256 * b;
#pragma unroll
            for (int s = 0; s < 8; ++s) {
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    const uint4 bfrag = *reinterpret_cast<const uint4*>(xb + boff[t] + kl[s]);
                    acc[t] = mfma16<DT>(a.operand(s), bfrag, acc[t]);
                }
            }
            if (++b == nb) {
                // C layout of 16x16x32: acc[t][v] = (weight row 4g + v, token 16t + r)
                const uint32_t out_row = tile * 16 + 4 * g;
#pragma unroll
                for (int t = 0; t < TT; ++t) {
                    if (16u * t + r < mt) {
                        const size_t base = (size_t)out_token[t] * n + out_row;
                        if (y_dtype == FH_F32 && (n & 3u) == 0 && out_row + 3 < n) {
                            *reinterpret_cast<float4*>(static_cast<float*>(ydst) + base) =
                                make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
                        } else if (y_dtype != FH_F32 && (n & 3u) == 0 && out_row + 3 < n) {
                            uint2 packed;
                            if (y_dtype == FH_F16) {
                                packed.x = f32_to_f16_bits(acc[t][0]) | (f32_to_f16_bits(acc[t][1]) << 16);
                                packed.y = f32_to_f16_bits(acc[t][2]) | (f32_to_f16_bits(acc[t][3]) << 16);
                            } else {
                                packed.x = f32_pair_to_bf16_bits(acc[t][0], acc[t][1]);
                                packed.y = f32_pair_to_bf16_bits(acc[t][2], acc[t][3]);
                            }
                            *reinterpret_cast<uint2*>(static_cast<uint16_t*>(ydst) + base) = packed;
                        } else {
#pragma unroll
                            for (int v = 0; v < 4; ++v)
                                if (out_row + v < n) store_from_f32(ydst, base + v, y_dtype, acc[t][v]);
                        }
                    }
                    acc[t] = float4v{0.f, 0.f, 0.f, 0.f};
                }
                b = 0;
                tile += kResWaves;
            }
        };
        uint32_t u = 0;
        for (; u + kResRing <= units; u += kResRing) {
#pragma unroll
            for (int i = 0; i < kResRing; ++i) {
                __builtin_amdgcn_sched_barrier(0);
                consume(ring[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < kResRing - 1; ++i)
            if (u + i < units) consume(ring[i]);
    }
}

// expert_resident_kernel with the weights going through LDS.  Loading weights straight into the
// MFMA operand layout puts sixteen different rows under sixteen neighbouring lanes, and the vector
// L1 then looks up one line per lane: the weight stream of that kernel stops at 3.4 TB/s.  A 16-row
// tile of weights is one contiguous run of 16 x nb x 144 bytes, so here every wave copies its tiles
// into a ring of LDS slots of its own with LDS-direct loads -- whole kilobytes per instruction, the
// next tiles on their way while this one is multiplied -- and the lanes pick their header and their
// chunk's quants out of LDS.  It needs room for the rings beside the token rows (rows of up to
// ~1024 weights for 32 tokens), and n a multiple of 16 (a tile is read whole).  Q4_K and Q6_K (a
// tile of either is a whole number of 16-byte pieces at a 16-byte aligned address).
template <uint32_t TYPE, int DT, int TT, int NB, bool F32>
__global__ __launch_bounds__(kResThreads) void expert_ring_kernel(const uint8_t* __restrict__ w,
                                                                 const uint16_t* __restrict__ x,
                                                                 void* __restrict__ y, uint32_t n,
                                                                 uint32_t nb, uint32_t y_dtype,
                                                                 const uint32_t* __restrict__ offsets,
                                                                 const uint32_t* __restrict__ order,
                                                                 uint32_t tiles_per_wg,
                                                                 const float* __restrict__ metadata,
                                                                 uint32_t x_rows, uint32_t routes,
                                                                 const ResidentShared sh, uint32_t ring_tiles) {
    constexpr uint32_t kBB = Quarter<TYPE>::kBlockBytes;
    constexpr int kTokens = 16 * TT;
    extern __shared__ __attribute__((aligned(16))) uint16_t xs[];

    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r = lane & 15u, g = lane >> 4;
    const uint32_t k = nb * 256, ld = k;
    const uint32_t expert_first = offsets != nullptr ? min(offsets[blockIdx.y], routes) : 0;
    const uint32_t expert_upto = offsets != nullptr ? min(offsets[blockIdx.y + 1], routes) : 0;
    const uint32_t count = expert_upto > expert_first ? expert_upto - expert_first : 0;
    const uint32_t tiles = n / 16;
    const uint32_t pieces = k / 8;  // 16-byte pieces per activation row
    // a tile of weights: 16 rows x nb super-blocks, contiguous; its ring slot, in whole kilobytes of requests
    const uint32_t tile_bytes = 16u * nb * kBB, per_tile = (tile_bytes + 1023u) >> 10;
    uint8_t* const ring = reinterpret_cast<uint8_t*>(xs) + (size_t)kTokens * k * 2 + (size_t)wave * ring_tiles * tile_bytes;
    const uint32_t ring_addr = (uint32_t)(uintptr_t)ring;

    const uint32_t passes = (count + kTokens - 1) / kTokens;
    const uint32_t wg = blockIdx.y * gridDim.x + blockIdx.x, wgs = gridDim.x * gridDim.y;
    const uint32_t shared_pieces = sh.w != nullptr ? (sh.tokens + kTokens - 1) / kTokens * sh.slices : 0;
    const uint32_t my_pieces = shared_pieces > wg ? (shared_pieces - wg + wgs - 1) / wgs : 0;
    for (uint32_t item = 0; item < passes + my_pieces; ++item) {
        const bool shared = item >= passes;  // uniform over the workgroup
        uint32_t first_token, mt, tile_begin, tile_end;
        if (!shared) {
            first_token = expert_first + item * kTokens;
            mt = min((uint32_t)kTokens, count - item * kTokens);
            tile_begin = blockIdx.x * tiles_per_wg + wave;
            tile_end = min(tiles, (blockIdx.x + 1) * tiles_per_wg);
        } else {
            const uint32_t piece = wg + (item - passes) * wgs;
            const uint32_t group = piece / sh.slices, slice = piece - group * sh.slices;
            first_token = group * kTokens;
            mt = min((uint32_t)kTokens, sh.tokens - first_token);
            tile_begin = slice * sh.tiles_per_slice + wave;
            tile_end = min(tiles, (slice + 1) * sh.tiles_per_slice);
        }
        const uint8_t* wexpert = shared ? sh.w : w + (size_t)blockIdx.y * n * nb * kBB;
        const uint16_t* xsrc = shared && sh.x != nullptr ? sh.x : x;
        void* ydst = shared ? sh.y : y;
        if (item != 0) __syncthreads();  // the previous item is done with the rows
        // this wave's tiles: tile_begin, tile_begin + 8, ..; the first ones are requested once the rows are
        // in LDS (the gather's own loads are the compiler's, and nothing of its may stand between a
        // request and the wait that counts it)
        const uint32_t my_tiles = tile_begin < tile_end ? (tile_end - tile_begin + kResWaves - 1) / kResWaves : 0;
        uint32_t requested = 0;
        auto request_tile = [&]() {
            const uint8_t* const base = wexpert + (size_t)(tile_begin + requested * kResWaves) * tile_bytes;
            const uint32_t slot_addr = ring_addr + (requested % ring_tiles) * tile_bytes;
            for (uint32_t c = 0; c < per_tile; ++c) {
                if (c * 1024u + lane * 16u < tile_bytes) lds_load16_at(base + c * 1024u, lane * 16u, slot_addr + c * 1024u);
            }
            ++requested;
        };
        gather_rows<F32>(xs, xsrc, mt, pieces, k, ld, first_token, shared ? nullptr : order, shared ? nullptr : metadata,
                    x_rows, tid);
        __syncthreads();
        if (my_tiles == 0) continue;  // uniform per wave; no barrier follows in this item

        // B operand rows: token 16t + r, clamped (columns past mt are never stored)
        uint32_t boff[TT];
        uint32_t out_token[TT];
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const uint32_t tok = min(16u * t + r, mt - 1);
            boff[t] = tok * ld;
            out_token[t] = order != nullptr && !shared ? order[first_token + tok] : first_token + tok;
        }
        // (the loads above are the last of the compiler's before the requests: it waits for them here,
        // where nothing of this wave's is in flight)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int t = 0; t < TT; ++t) asm volatile("" : "+v"(out_token[t]));
        while (requested < my_tiles && requested < ring_tiles) request_tile();
        uint32_t kl[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) kl[s] = (((Quarter<TYPE>::klocal(g, s) >> 3) ^ r) << 3);  // row 16t + r: swizzle r

        // Every tile multiplies the same token rows.  Where they fit the wave's registers (two waves a
        // SIMD leave each 256) the B operands are read out of LDS once per item and not once per tile:
        // read per tile they are 16 KB per wave and super-block, more LDS traffic than the weights
        // (32 registers per super-block and 16 tokens)
        constexpr bool kRowsInRegisters = NB * TT <= 4 && TYPE == kQ4K;
        uint4 brow[kRowsInRegisters ? NB * 8 * TT : 1];
        if constexpr (kRowsInRegisters) {
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int s = 0; s < 8; ++s)
#pragma unroll
                    for (int t = 0; t < TT; ++t)
                        brow[(b * 8 + s) * TT + t] = *reinterpret_cast<const uint4*>(xs + 256 * b + boff[t] + kl[s]);
        }

        float4v acc[TT];
#pragma unroll
        for (int t = 0; t < TT; ++t) acc[t] = float4v{0.f, 0.f, 0.f, 0.f};
        // lane (r, g) finds row r of a slot at r x nb x 144
        const uint32_t lane_row = r * nb * kBB;
        for (uint32_t i = 0; i < my_tiles; ++i) {
            const uint32_t tile = tile_begin + i * kResWaves;
            // requests retire in issue order: behind tile i's stand those of the tiles asked for since
            wait_vmcnt((requested - 1u - i) * per_tile);
            const uint8_t* const slot = ring + (i % ring_tiles) * tile_bytes + lane_row;
            // the whole tile (NB super-blocks of the lane's row) leaves its slot at once, and the slot
            // is asked for the tile `ring_tiles` places ahead before anything is multiplied: a slot is
            // out of flight for one LDS round trip, not for a tile's arithmetic.  (Reading tile i + 1
            // out of LDS while tile i is multiplied takes that round trip out of the wave's way too and
            // changes nothing: the kernel is bound by its decode arithmetic.)
            Quarter<TYPE> q[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                // Rows of an even number of 210-byte blocks begin at a dword, every other block between two, where LDS takes longer
                // for 16 bytes than for the two aligned reads that cover them (us, routed FFN of 256 experts, Q4_K with Q6_K 2048 x 512
                // down, 200 / 512 / 1024 tokens: 224 / 195 / 343, so 208 / 184 / 320).  (Where rows are of an odd number the lanes
                // differ.)
                if constexpr (TYPE == kQ6K && NB % 2 == 0) q[b].load_by_dwords(slot + b * kBB, g, (b & 1) != 0);
                else q[b].load(slot + b * kBB, g);
            }
            if (requested < my_tiles) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                request_tile();
            }
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                PackedOperands<DT> a;
                q[b].decode_into(g, a);
                const uint16_t* xb = xs + 256 * b;
#pragma unroll
                for (int s = 0; s < 8; ++s) {
#pragma unroll
                    for (int t = 0; t < TT; ++t) {
                        uint4 bfrag;
                        if constexpr (kRowsInRegisters) bfrag = brow[(b * 8 + s) * TT + t];
                        else bfrag = *reinterpret_cast<const uint4*>(xb + boff[t] + kl[s]);
                        acc[t] = mfma16<DT>(a.operand(s), bfrag, acc[t]);
                    }
                }
            }
            // C layout of 16x16x32: acc[t][v] = (weight row 4g + v, token 16t + r)
            const uint32_t out_row = tile * 16 + 4 * g;
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                if (16u * t + r < mt) {
                    const size_t base = (size_t)out_token[t] * n + out_row;
                    if (y_dtype == FH_F32) {
                        *reinterpret_cast<float4*>(static_cast<float*>(ydst) + base) =
                            make_float4(acc[t][0], acc[t][1], acc[t][2], acc[t][3]);
                    } else {
                        uint2 packed;
                        if (y_dtype == FH_F16) {
                            packed.x = f32_to_f16_bits(acc[t][0]) | (f32_to_f16_bits(acc[t][1]) << 16);
                            packed.y = f32_to_f16_bits(acc[t][2]) | (f32_to_f16_bits(acc[t][3]) << 16);
                        } else {
                            packed.x = f32_pair_to_bf16_bits(acc[t][0], acc[t][1]);
                            packed.y = f32_pair_to_bf16_bits(acc[t][2], acc[t][3]);
                        }
                        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(ydst) + base) = packed;
                    }
                }
                acc[t] = float4v{0.f, 0.f, 0.f, 0.f};
            }
        }
        // (the last tile's wait left none of this wave's requests in flight; said where the next
        // item's loads can see it)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
}

// Tokens an expert's workgroup takes in one pass over its weights: 32 with more than 8 per expert on average,
// else 16, unless 32 rows fit LDS and one expert is likely enough to have more than 16: its second pass nearly
// doubles the launch (256 experts top-8, 256 tokens 209 us in passes of 16, 158 in passes of 32), where
// passes of 32 cost 5 - 14% (256 experts of 1024 x 2048, 200 tokens: IQ4_XS 106 us and 121, Q8_0 133 and 150).  Ids
// drawn evenly, the counts are close to Poisson's; the line at a chance of a fifth is 6.9 tokens per expert
// for 256 of them, 7.3 for 128, 7.9 for 64.
bool passes_of_32(uint32_t k, uint32_t m, uint32_t experts) {
    if (m > 8 * experts) return true;
    if (m <= 6 * experts || (size_t)32 * k * 2 > kResLdsBytes) return false;
    const double mean = (double)m / (double)experts;
    double term = std::exp(-mean), up_to_16 = term;
    for (int i = 1; i <= 16; ++i) up_to_16 += term *= mean / i;
    return experts * (1.0 - up_to_16) > 0.2;
}

template <uint32_t TYPE, int DT>
void launch_tt(hipStream_t s, const GemmArgs& a) {
    const uint8_t* w = static_cast<const uint8_t*>(a.w);
    const uint16_t* x = static_cast<const uint16_t*>(a.x);
    const uint32_t nb = a.k / 256;
    if (a.use_resident) {
        // dense product with the activation rows resident in LDS: (32-row group, row-tile slice)
        // pieces, about one per compute unit
        const bool wide = a.m > 16 && (size_t)32 * a.k * 2 <= kResLdsBytes;
        const uint32_t per_group = wide ? 32u : 16u;
        const size_t lds = (size_t)per_group * a.k * 2;
        const uint32_t tiles = (a.n + 15) / 16;
        const uint32_t cus = a.cu_count > 0 ? (uint32_t)a.cu_count : 256u;
        const uint32_t groups = (a.m + per_group - 1) / per_group;
        // never a few pieces more than workgroups: those would make a second round
        const uint32_t want = cus / groups > 0 ? cus / groups : 1;
        ResidentShared sh{};
        sh.w = w;
        sh.x = nullptr;
        sh.y = a.y;
        sh.tokens = a.m;
        sh.tiles_per_slice = (tiles + want - 1) / want;
        sh.slices = (tiles + sh.tiles_per_slice - 1) / sh.tiles_per_slice;
        const uint32_t pieces = groups * sh.slices;
        const dim3 rgrid(pieces < cus ? pieces : cus, 1);
        if (wide) {
            auto kernel = expert_resident_kernel<TYPE, DT, 2>;
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            hipLaunchKernelGGL(kernel, rgrid, dim3(kResThreads), lds, s, nullptr, x, nullptr, a.n, nb, a.y_dtype,
                               nullptr, nullptr, 0u, nullptr, 0u, 0u, sh);
        } else {
            auto kernel = expert_resident_kernel<TYPE, DT, 1>;
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            hipLaunchKernelGGL(kernel, rgrid, dim3(kResThreads), lds, s, nullptr, x, nullptr, a.n, nb, a.y_dtype,
                               nullptr, nullptr, 0u, nullptr, 0u, 0u, sh);
        }
        return;
    }
    const bool wide = passes_of_32(a.k, a.m, a.experts);
    const size_t lds = (size_t)(wide ? 32 : 16) * a.k * 2;
    if (expert_rows_fit_lds(a.k, a.m, a.experts)) {
        // An expert's rows are cut into shares so that about one workgroup per compute unit has work.
        // Every share gathers the expert's tokens again: with all of 256 experts hit one share each
        // (236 us for the 512-token routed FFN) beats four (264).  With fewer assignments than experts
        // the compute units of those that nobody chose would idle: the hit ones, were the ids drawn
        // evenly, share the chip (256 experts top-8, 4 / 8 / 16 tokens: 116 / 117 / 118 us with one
        // share, 62 / 80 / 102 with four).  Two deviations more than the mean count as hit: a workgroup
        // over the chip's number is a round of its own (64 experts of 2816 x 2048 Q6_K, 96 assignments to 53 of
        // them: 107 us in five shares, 92 in four).  Below twice the shares that all experts would get it does not
        // pay: the workgroups of the others also carry the shared expert's pieces (64 experts of 2048 x 1024 and a
        // shared one, five tokens top-8: Q6_K 48 - 60 us in six or eight shares, 42 in four).
        const uint32_t tiles = (a.n + 15) / 16;
        const uint32_t target = a.cu_count > 0 ? (uint32_t)a.cu_count : 256u;
        const double missed = std::pow(1.0 - 1.0 / (double)a.experts, (double)a.m);
        const double hit = std::min({(double)a.experts, (double)a.m,
                                     a.experts * (1.0 - missed) + 2.0 * std::sqrt(a.experts * missed * (1.0 - missed))});
        const uint32_t all_hit = (target + a.experts - 1) / a.experts, few_hit = (uint32_t)(target / std::max(hit, 1.0));
        const uint32_t shares = few_hit >= 2 * all_hit ? few_hit : all_hit;
        uint32_t tiles_per_wg = (tiles + shares - 1) / shares;
        tiles_per_wg = (tiles_per_wg + kResWaves - 1) / kResWaves * kResWaves;
        const dim3 rgrid((tiles + tiles_per_wg - 1) / tiles_per_wg, a.experts);
        ResidentShared sh{};
        if (a.shared_w != nullptr) {
            sh.w = static_cast<const uint8_t*>(a.shared_w);
            sh.x = static_cast<const uint16_t*>(a.shared_x);
            sh.y = a.shared_y;
            sh.tokens = a.shared_rows;
            // about one piece per workgroup: a token group's rows are cut into as many slices
            const uint32_t per_group = wide ? 32u : 16u;
            const uint32_t groups = (a.shared_rows + per_group - 1) / per_group;
            const uint32_t want = rgrid.x * rgrid.y / groups > 0 ? rgrid.x * rgrid.y / groups : 1;
            sh.tiles_per_slice = (tiles + want - 1) / want;
            sh.slices = (tiles + sh.tiles_per_slice - 1) / sh.tiles_per_slice;
        }
        // weights through rings in LDS where those fit beside the rows (short rows: the down projections)
        // (Q4_K 49 against 55 us and Q6_K 74 against 77 for 256 experts x 2048 x 512 over 4096 rows; IQ4_XS,
        // whose rows' operands do not fit the registers beside its decode, 62 either way: it stays)
        auto launch = [&](auto rounds) {
            constexpr bool kF32 = DT == 1 && decltype(rounds)::value;
            if constexpr (TYPE == kQ4K || TYPE == kQ6K) {
                const size_t tile_bytes = (size_t)16 * nb * Quarter<TYPE>::kBlockBytes;
                const size_t room = kResLdsBytes > lds ? (kResLdsBytes - lds) / (kResWaves * tile_bytes) : 0;
                const uint32_t ring_tiles = room >= 3 ? 3u : (uint32_t)room;
                if (a.weight_ring && a.n % 16 == 0 && nb <= 4 && ring_tiles >= 2) {
                    const size_t ring_lds = lds + kResWaves * ring_tiles * tile_bytes;
                    typedef void (*Ring)(const uint8_t*, const uint16_t*, void*, uint32_t, uint32_t, uint32_t,
                                         const uint32_t*, const uint32_t*, uint32_t, const float*, uint32_t, uint32_t,
                                         const ResidentShared, uint32_t);
                    static const Ring rings[2][4] = {
                        {expert_ring_kernel<TYPE, DT, 1, 1, kF32>, expert_ring_kernel<TYPE, DT, 1, 2, kF32>,
                         expert_ring_kernel<TYPE, DT, 1, 3, kF32>, expert_ring_kernel<TYPE, DT, 1, 4, kF32>},
                        {expert_ring_kernel<TYPE, DT, 2, 1, kF32>, expert_ring_kernel<TYPE, DT, 2, 2, kF32>,
                         expert_ring_kernel<TYPE, DT, 2, 3, kF32>, expert_ring_kernel<TYPE, DT, 2, 4, kF32>}};
                    const Ring kernel = rings[wide ? 1 : 0][nb - 1];
                    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)ring_lds);
                    hipLaunchKernelGGL(kernel, rgrid, dim3(kResThreads), ring_lds, s, w, x, a.y, a.n, nb, a.y_dtype,
                                       a.expert_offsets, a.expert_order, tiles_per_wg, a.gather_metadata, a.x_rows, a.m,
                                       sh, ring_tiles);
                    return;
                }
            }
            auto kernel = wide ? expert_resident_kernel<TYPE, DT, 2, kF32> : expert_resident_kernel<TYPE, DT, 1, kF32>;
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)lds);
            hipLaunchKernelGGL(kernel, rgrid, dim3(kResThreads), lds, s, w, x, a.y, a.n, nb, a.y_dtype,
                               a.expert_offsets, a.expert_order, tiles_per_wg, a.gather_metadata, a.x_rows, a.m, sh);
        };
        if (DT == 1 && a.x_rounds) launch(std::true_type{});
        else launch(std::false_type{});
        return;
    }
    const dim3 grid((a.n + kSkRows - 1) / kSkRows, a.experts);
    if (!wide) {
        hipLaunchKernelGGL((gemm_skinny_kernel<TYPE, DT, 1>), grid, dim3(kSkThreads), 0, s, w, x,
                           a.y, a.m, a.n, nb, a.y_dtype, a.expert_offsets, a.expert_order);
    } else {
        hipLaunchKernelGGL((gemm_skinny_kernel<TYPE, DT, 2>), grid, dim3(kSkThreads), 0, s, w, x,
                           a.y, a.m, a.n, nb, a.y_dtype, a.expert_offsets, a.expert_order);
    }
    return;
}

}  // namespace

bool expert_rows_fit_lds(uint32_t k, uint32_t m, uint32_t experts) {
    return (size_t)(passes_of_32(k, m, experts) ? 32 : 16) * k * 2 <= kResLdsBytes;
}

const char* launch_gemm_resident(hipStream_t s, const GemmArgs& dense) {
    GemmArgs a = dense;
    a.use_resident = true;
    a.expert_offsets = nullptr;
    {
        static const char* const names[5] = {"q4_k_gemm_mfma_resident", "q5_k_gemm_mfma_resident",
                                             "q6_k_gemm_mfma_resident", "iq4_xs_gemm_mfma_resident",
                                             "q8_0_gemm_mfma_resident"};
        const int f = a.ggml_type == kQ4K ? 0 : a.ggml_type == kQ5K ? 1 : a.ggml_type == kQ6K ? 2 : a.ggml_type == kIQ4XS ? 3 : 4;
#define FH_RES(TYPE) \
    if (a.x_dtype == FH_F16) launch_tt<TYPE, 1>(s, a); else launch_tt<TYPE, 2>(s, a)
        if (f == 0) { FH_RES(kQ4K); } else if (f == 1) { FH_RES(kQ5K); } else if (f == 2) { FH_RES(kQ6K); }
        else if (f == 3) { FH_RES(kIQ4XS); } else { FH_RES(kQ8_0); }
#undef FH_RES
        return names[f];
    }
}

const char* launch_gemm_skinny(hipStream_t s, const GemmArgs& a) {
    if (a.ggml_type == kQ4K) {
        if (a.x_dtype == FH_F16) launch_tt<kQ4K, 1>(s, a); else launch_tt<kQ4K, 2>(s, a);
        return "expert_project_q4_k_grouped_mfma";
    }
    if (a.ggml_type == kQ5K) {
        if (a.x_dtype == FH_F16) launch_tt<kQ5K, 1>(s, a); else launch_tt<kQ5K, 2>(s, a);
        return "expert_project_q5_k_grouped_mfma";
    }
    if (a.ggml_type == kIQ4XS) {
        if (a.x_dtype == FH_F16) launch_tt<kIQ4XS, 1>(s, a); else launch_tt<kIQ4XS, 2>(s, a);
        return "expert_project_iq4_xs_grouped_mfma";
    }
    if (a.ggml_type == kQ8_0) {
        if (a.x_dtype == FH_F16) launch_tt<kQ8_0, 1>(s, a); else launch_tt<kQ8_0, 2>(s, a);
        return "expert_project_q8_0_grouped_mfma";
    }
    if (a.x_dtype == FH_F16) launch_tt<kQ6K, 1>(s, a); else launch_tt<kQ6K, 2>(s, a);
    return "expert_project_q6_k_grouped_mfma";
}

}  // namespace fh
