// Projection of a few rows, Y[M,N] = X[M,K] . W[N,K]^T for Q4_K / Q5_K / Q6_K / IQ4_XS / Q8_0
// weights, on the matrix cores: f16 / bf16 rows with weights rounded once to the row's type
// (v_mfma_f32_16x16x32), or f32 rows with exact f32 weights (v_mfma_f32_16x16x4_f32).
//
// With this few rows the job is a weight stream.  Every wave owns a set of super-blocks along K and
// multiplies them by all of its workgroup's weight tiles (16 rows each): the activations of one
// super-block become matrix operands in registers once and serve every tile, the raw weights of the
// next super-block are requested tile by tile as this one's are decoded, and the only barrier is at
// the end, where the waves' partial sums meet in LDS (added in wave order: deterministic).  Nothing
// depends on the length of a row, so any K runs; few tiles and long rows are cut into K segments
// across workgroups, whose partial sums meet in device memory and are added in segment order by the
// last workgroup to arrive.
//
// Activations travel as whole cache lines straight into a piece of LDS that belongs to the wave
// (buffer_load .. lds, 16 bytes a lane) and from there into operand order; loading operands from
// memory as they are used would touch one line per lane.  They are requested one super-block ahead,
// like the weights: loads return in order, so a nearer request would wait for the farther ones.
#pragma once

#include <hip/hip_runtime.h>
#include <type_traits>

#include "device_utils.hpp"
#include "internal.hpp"
#include "lds_direct.hpp"
#include "quarter.hpp"
#include "tile_decode.hpp"

namespace fh {

struct RowsParams {
    const uint8_t* w;
    const uint8_t* x;
    void* y;
    uint32_t m, n, nb;
    uint32_t y_dtype;
    uint32_t k_waves;      // waves that share a tile's super-blocks: 8 / k_waves sets of tiles per workgroup
    uint32_t groups;       // groups of 16 * TT rows
    uint32_t tile_groups;  // groups of T * 8 / k_waves weight tiles
    uint32_t segments, seg_blocks;
    float* partials;       // [segments][m][n]
    uint32_t* counters;    // one per (tile group, row group), zero between launches
};

// one per format, each in a source file of its own (gemm_rows_<format>.hip): two hundred kernels are
// too many for one compilation
void launch_rows_q4_k(hipStream_t s, uint32_t dtype, const RowsPlan& plan, const RowsParams& p);
void launch_rows_q5_k(hipStream_t s, uint32_t dtype, const RowsPlan& plan, const RowsParams& p);
void launch_rows_q6_k(hipStream_t s, uint32_t dtype, const RowsPlan& plan, const RowsParams& p);
void launch_rows_iq4_xs(hipStream_t s, uint32_t dtype, const RowsPlan& plan, const RowsParams& p);
void launch_rows_q8_0(hipStream_t s, uint32_t dtype, const RowsPlan& plan, const RowsParams& p);

namespace {

constexpr int kRowsWaves = 8;
constexpr uint32_t kRowsThreads = 64 * kRowsWaves;

template <int DT>
constexpr uint32_t kXRowBytes = DT == 0 ? 1024u : 512u;   // a row's share of a super-block

template <int DT, int ROWS>
constexpr uint32_t kWaveLds = (uint32_t)ROWS * kXRowBytes<DT>;

// Steps FROM .. FROM + COUNT of a super-block of exact f32 operands.  Four steps are chained in the
// accumulator (16 roundings one after the other), the rest is added in pairs: with all 64 steps in one
// chain the product was up to four times as far from 64 bits as the GEMV kernels are (rel-L2 of 64 x 777 x
// 5120 Q5_K 4.5e-7, now 1.12e-7, the GEMV 1.11e-7; 16 x 1024 x 1024 Q4_K 2.8e-7, 1.00e-7, 1.02e-7).  It costs
// a tenth: a block of projections over 24 rows 213 us, 195 in one chain, 585 on the GEMV.
template <int FROM, int COUNT>
__device__ __forceinline__ float4v pairwise(const FloatOperands& a, const u32x4 (&x)[16]) {
    if constexpr (COUNT > 4) {
        const float4v lo = pairwise<FROM, COUNT / 2>(a, x);
        return lo + pairwise<FROM + COUNT / 2, COUNT / 2>(a, x);
    } else {
        float4v sum{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = FROM; s < FROM + COUNT; ++s)
            sum = __builtin_amdgcn_mfma_f32_16x16x4f32(a.v[s], __uint_as_float(x[s >> 2][s & 3]), sum, 0, 0, 0);
        return sum;
    }
}

// ROWS: activation rows of a workgroup, 16 or 32 (a slab of 8 for up to 8 rows measured 17.0 against
// 17.3 us at 8 x 17408 x 5120: not worth a third more kernels); T: weight tiles per wave.
// A workgroup has one item of work and a compute unit one workgroup (the operands of a super-block,
// a raw tile ahead for every tile and the sums take the registers of two waves a SIMD).  Walking
// several items per workgroup with the next one's weights already on their way was measured: large
// matrices 5 - 15% faster at 16 rows (65536 x 5120 50.7 against 56.6 us), everything at 32 rows 10 -
// 35% slower (17408 x 5120 28.9 against 21.2: the extra registers spill).
template <uint32_t TYPE, int DT, int ROWS, int T>
__global__ __launch_bounds__(kRowsThreads) void gemm_rows_kernel(const RowsParams p) {
    constexpr int TT = ROWS / 16;                                   // 16-column operands
    constexpr uint32_t kBB = Quarter<TYPE>::kBlockBytes;
    constexpr uint32_t kRowBytes = kXRowBytes<DT>;
    constexpr uint32_t kTokensPerLoad = 1024u / kRowBytes;          // rows one 1 KB request covers
    constexpr int kLoads = (int)(ROWS / kTokensPerLoad);
    constexpr int kFrags = DT == 0 ? 16 : 8;                        // 16-byte operand pieces per lane, block and 16 rows
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ uint32_t last_flag;

    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t r = lane & 15u, g = lane >> 4;

    const uint32_t tile_waves = kRowsWaves / p.k_waves;
    const uint32_t k_wave = wave % p.k_waves, tile_wave = wave / p.k_waves;

    // ids that are equal mod 8 sit on one XCD: the row groups of a tile group share its weights in that L2
    uint32_t tile_group, group;
    {
        const uint32_t per = 8u * p.groups, q = blockIdx.x / per, rest = blockIdx.x - q * per;
        tile_group = 8u * q + (rest & 7u);
        group = rest >> 3;
        if (tile_group >= p.tile_groups) return;
    }
    const uint32_t group_tile0 = tile_group * T * tile_waves, tile0 = group_tile0 + tile_wave * T;
    const uint32_t b0 = blockIdx.y * p.seg_blocks + k_wave, end = min(p.nb, (blockIdx.y + 1u) * p.seg_blocks);
    const uint32_t m0 = group * ROWS, mt = min((uint32_t)ROWS, p.m - m0);
    float4v acc[T][TT];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < TT; ++i) acc[t][i] = float4v{0.f, 0.f, 0.f, 0.f};

    if (b0 < end) {
        // weight rows past the matrix re-read its last one; what they produce is never stored
        const uint8_t* wrow[T];
#pragma unroll
        for (int t = 0; t < T; ++t) wrow[t] = p.w + (size_t)min((tile0 + t) * 16 + r, p.n - 1) * p.nb * kBB;
        // request j of a block brings rows kTokensPerLoad * j ..; the 16-byte piece c of row t lands at
        // piece c ^ (t & 15), so that the sixteen rows an operand read touches fall on different banks.  (Rows past the
        // batch lie past the buffer, without traffic: the columns they would feed are never stored.  The descriptor and the rows'
        // offsets are made behind the first loads and only for waves with more than one super-block: 57 x 665 x 1024 takes
        // 4.5 us, and 4.8 where they stand ahead of the first requests.)
        uint8_t* const slab = lds + wave * kWaveLds<DT, ROWS>;
        const uint32_t x_row = p.nb * kRowBytes;
        const uint32_t sub = DT == 0 ? 0u : lane >> 5, piece = DT == 0 ? lane : lane & 31u;
        Quarter<TYPE> raw[T];
        // the first ones, ahead of every load that the compiler counts (and of every M0 that it writes), by hand
        const uint8_t* const first_rows = p.x + (size_t)m0 * x_row + (size_t)b0 * kRowBytes;
        const uint32_t slab_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)slab;
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const uint32_t tok = (uint32_t)j * kTokensPerLoad + sub;
            lds_load16_uniform(first_rows, min(tok, mt - 1) * x_row + 16u * (piece ^ (tok & 15u)), slab_at + 1024u * j);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < T; ++t) {
            raw[t].load(wrow[t] + (size_t)b0 * kBB, g);
            __builtin_amdgcn_sched_barrier(0);
        }
        auto block = [&](uint32_t b, auto more, auto&& request_rows) {
            constexpr bool kMore = decltype(more)::value;
            // This block's rows have landed once no more than the T tiles' weight requests behind them are
            // outstanding (loads retire in order).  The compiler counts its own waits with these requests in
            // sight but puts none of its own before the reads of what they write; the build counts the loads
            // between the two in the generated code (ferrum_amd/isa_check.py).  (Requested by the builtin for global
            // loads, which is a flat access to the compiler, they made it wait for everything outstanding before the first
            // tile of every super-block.  us then / now: 64 x 5120 x 17408 44.1 / 42.7, Q6_K
            // 32 x 5120 x 17408 38.1 / 34.9, Q4_K 16 x 28672 x 4096 27.8 / 24.9 where it is asked to take it; 36 drawn products
            // 1.04 x in the mean: profiles/waits_loads_lookups_us.txt.)
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(T * Quarter<TYPE>::kLoads) : "memory");
            u32x4 frag[TT][kFrags];
#pragma unroll
            for (int i = 0; i < TT; ++i)
#pragma unroll
                for (int s = 0; s < kFrags; ++s) {
                    const uint32_t kl = DT == 0 ? (Quarter<TYPE>::klocal(g, s >> 1) >> 2) + (s & 1u)
                                                : Quarter<TYPE>::klocal(g, s) >> 3;
                    frag[i][s] = *reinterpret_cast<const u32x4*>(slab + (16 * i + r) * kRowBytes + 16 * (kl ^ r));
                }
            if constexpr (kMore) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the operands have left the slab
                request_rows(b + p.k_waves);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < T; ++t) {
                if constexpr (DT == 0) {
                    FloatOperands a;
                    raw[t].decode_into(g, a);
                    if constexpr (kMore) raw[t].load(wrow[t] + (size_t)(b + p.k_waves) * kBB, g);
#pragma unroll
                    for (int i = 0; i < TT; ++i) acc[t][i] += pairwise<0, 64>(a, frag[i]);
                } else {
                    PackedOperands<DT> a;
                    raw[t].decode_into(g, a);
                    if constexpr (kMore) raw[t].load(wrow[t] + (size_t)(b + p.k_waves) * kBB, g);
#pragma unroll
                    for (int s = 0; s < 8; ++s)
#pragma unroll
                        for (int i = 0; i < TT; ++i)
                            acc[t][i] = mfma16<DT>(a.operand(s), __builtin_bit_cast(uint4, frag[i][s]), acc[t][i]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        uint32_t b = b0;
        if (b + p.k_waves < end) {
            const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
                reinterpret_cast<void*>(uniform_address(p.x + (size_t)m0 * x_row)), 0, mt * x_row, 0x00027000);
            uint32_t row_at[kLoads];
#pragma unroll
            for (int j = 0; j < kLoads; ++j) {
                const uint32_t tok = (uint32_t)j * kTokensPerLoad + sub;
                row_at[j] = tok < mt ? tok * x_row + 16u * (piece ^ (tok & 15u)) : kRowsBatchBytes;
            }
            auto request_rows = [&](uint32_t of) {
#pragma unroll
                for (int j = 0; j < kLoads; ++j) lds_load16_counted(rows, slab + 1024 * j, row_at[j], of * kRowBytes);
            };
            do {
                block(b, std::true_type{}, request_rows);
                b += p.k_waves;
            } while (b + p.k_waves < end);
        }
        block(b, std::false_type{}, [](uint32_t) {});
    }

    // the waves' partial sums, in the place of the activations
    __syncthreads();
    float4* const partial = reinterpret_cast<float4*>(lds);
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int i = 0; i < TT; ++i)
            partial[(((tile_wave * T + t) * TT + i) * p.k_waves + k_wave) * 64 + lane] =
                make_float4(acc[t][i][0], acc[t][i][1], acc[t][i][2], acc[t][i][3]);
    __syncthreads();
    // C layout of the 16x16 forms: lane (g, r) holds weight rows 4g .. 4g + 3 of token r.  Four rows
    // of a token per thread, neighbouring threads on neighbouring rows.
    const uint32_t quads = tile_waves * T * 4;
    const bool whole_quads = (p.n & 3u) == 0;
    auto each_quad = [&](auto&& body) {
        for (uint32_t idx = tid; idx < quads * mt; idx += kRowsThreads) {
            const uint32_t token = idx / quads, quad = idx - token * quads;
            const uint32_t row = group_tile0 * 16 + quad * 4;
            if (row < p.n) body(token, quad, row);
        }
    };
    auto store = [&](uint32_t token, uint32_t row, float4 v) {
        const size_t base = (size_t)(m0 + token) * p.n + row;
        if (whole_quads && p.y_dtype == FH_F32) {
            *reinterpret_cast<float4*>(static_cast<float*>(p.y) + base) = v;
        } else if (whole_quads) {
            const uint2 packed = p.y_dtype == FH_F16
                                     ? make_uint2(f32_to_f16_bits(v.x) | (f32_to_f16_bits(v.y) << 16),
                                                  f32_to_f16_bits(v.z) | (f32_to_f16_bits(v.w) << 16))
                                     : make_uint2(f32_pair_to_bf16_bits(v.x, v.y), f32_pair_to_bf16_bits(v.z, v.w));
            *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.y) + base) = packed;
        } else {
            const float vals[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (row + i < p.n) store_from_f32(p.y, base + i, p.y_dtype, vals[i]);
        }
    };
    each_quad([&](uint32_t token, uint32_t quad, uint32_t row) {
        const uint32_t at = (((quad >> 2) * TT + (token >> 4)) * p.k_waves) * 64 + (quad & 3u) * 16 + (token & 15u);
        float4 sum = partial[at];
        for (uint32_t k = 1; k < p.k_waves; ++k) {
            const float4 v = partial[at + k * 64];
            sum.x += v.x;
            sum.y += v.y;
            sum.z += v.z;
            sum.w += v.w;
        }
        if (p.segments == 1) {
            store(token, row, sum);
        } else {
            // device-scope accesses: coherent across the chip's L2 slices without cache-wide flushes
            float* const dst = p.partials + ((size_t)blockIdx.y * p.m + m0 + token) * p.n + row;
            const float vals[4] = {sum.x, sum.y, sum.z, sum.w};
            if (whole_quads) {
                typedef unsigned long long u64;
                u64* const d2 = reinterpret_cast<u64*>(dst);
                __hip_atomic_store(d2, (u64)__float_as_uint(sum.x) | ((u64)__float_as_uint(sum.y) << 32),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(d2 + 1, (u64)__float_as_uint(sum.z) | ((u64)__float_as_uint(sum.w) << 32),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (row + i < p.n) __hip_atomic_store(dst + i, vals[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    });
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
    each_quad([&](uint32_t token, uint32_t, uint32_t row) {
        float sum[4] = {0.f, 0.f, 0.f, 0.f};
        for (uint32_t s = 0; s < p.segments; ++s) {
            const float* const src = p.partials + ((size_t)s * p.m + m0 + token) * p.n + row;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (row + i < p.n) sum[i] += __hip_atomic_load(src + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        store(token, row, make_float4(sum[0], sum[1], sum[2], sum[3]));
    });
}

template <uint32_t TYPE, int DT, int ROWS, int T>
void launch_one(hipStream_t s, const RowsPlan& plan, const RowsParams& p) {
    constexpr uint32_t kSums = T * (ROWS / 16) * 1024u;   // partial sums of a wave
    constexpr size_t kLds = kRowsWaves * (kWaveLds<DT, ROWS> > kSums ? kWaveLds<DT, ROWS> : kSums);
    static std::atomic<uint64_t> raised{0};
    once_per_device(raised, [] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_rows_kernel<TYPE, DT, ROWS, T>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds);
    });
    hipLaunchKernelGGL((gemm_rows_kernel<TYPE, DT, ROWS, T>), dim3((p.tile_groups + 7) / 8 * 8 * p.groups, plan.segments),
                       dim3(kRowsThreads), kLds, s, p);
}

template <uint32_t TYPE, int DT, int ROWS>
void launch_tiles(hipStream_t s, const RowsPlan& plan, const RowsParams& p) {
    switch (plan.tiles) {
        case 1: return launch_one<TYPE, DT, ROWS, 1>(s, plan, p);
        case 2: return launch_one<TYPE, DT, ROWS, 2>(s, plan, p);
        case 3: return launch_one<TYPE, DT, ROWS, 3>(s, plan, p);
        case 4: return launch_one<TYPE, DT, ROWS, 4>(s, plan, p);
        default: return launch_one<TYPE, DT, ROWS, 5>(s, plan, p);
    }
}

template <uint32_t TYPE>
void launch_rows_of(hipStream_t s, uint32_t dtype, const RowsPlan& plan, const RowsParams& p) {
    if (dtype == FH_F32) launch_tiles<TYPE, 0, 16>(s, plan, p);
    else if (dtype == FH_F16 && plan.rows == 16) launch_tiles<TYPE, 1, 16>(s, plan, p);
    else if (dtype == FH_F16) launch_tiles<TYPE, 1, 32>(s, plan, p);
    else if (plan.rows == 16) launch_tiles<TYPE, 2, 16>(s, plan, p);
    else launch_tiles<TYPE, 2, 32>(s, plan, p);
}

}  // namespace
}  // namespace fh
