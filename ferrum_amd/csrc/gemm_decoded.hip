// Prefill in two passes: the weights of a panel of columns are decoded once into 16-bit tiles in the scratch, then
// multiplied by all rows, Y[M,N] = X[M,K] . W[N,K]^T, f16 or bf16, f32 accumulation.
//
// The tiles of gemm.hip decode every weight once per 256 rows beside the matrix cores; with many row tiles that is the
// same work again and again (Q8_0 1999 x 17408 x 5120: 560 us, 0.64 PFLOP/s; Q4_K 420).  Here the decode is a launch of its own, its bytes are the same
// (each weight the exact f32 value rounded once), and the product has nothing but matrix instructions, fragment reads and
// LDS-direct loads in its loop.
//
// A decoded panel lies as the product's LDS image: [32 columns][64 K] is four kilobytes, step s (0..3) a kilobyte of 64
// lanes x 8 weights, lane (c, kg) holding column c, K 32 (s / 2) + 16 kg + 8 (s % 2) ..  A workgroup's share of a slab is then whole
// kilobytes for LDS-direct loads, and a fragment read is 16 bytes a lane in lane order, free of bank conflicts.
#include <algorithm>
#include <type_traits>

#include "device_utils.hpp"
#include "internal.hpp"
#include "lds_direct.hpp"
#include "quarter.hpp"
#include "tile_decode.hpp"

namespace fh {
namespace {

typedef float float16v __attribute__((ext_vector_type(16)));

constexpr uint32_t kSlabTileBytes = 4096;   // 32 columns x 64 K

// A workgroup decodes kDecodeBlocks super-blocks of 32 columns, all requested before the first is decoded: two waves a
// super-block, a lane a quarter of one column's.  The tile goes through LDS and leaves as whole kilobytes in address order:
// stored from the lanes as they are, every wave of the chip writes pieces of 256 bytes four kilobytes apart, the same few
// memory channels at a time.  8192 x 5120 Q4_K 18 us, 5.9 TB/s.
constexpr uint32_t kDecodeBlocks = 4;
template <uint32_t TYPE, int DT>
__global__ __launch_bounds__(256) void decode_panel_kernel(const uint8_t* __restrict__ w, uint8_t* __restrict__ out, uint32_t n,
                                                           uint32_t nb) {
    __shared__ __attribute__((aligned(16))) uint8_t image[2][4 * kSlabTileBytes];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, r = lane & 15u, g = lane >> 4;
    const uint32_t b0 = blockIdx.x * kDecodeBlocks + (wave >> 1), tile = blockIdx.y, column = (wave & 1u) * 16 + r;
    const uint8_t* const row = w + (size_t)min(tile * 32 + column, n - 1) * nb * Quarter<TYPE>::kBlockBytes;
    Quarter<TYPE> raw[kDecodeBlocks / 2];
#pragma unroll
    for (uint32_t i = 0; i < kDecodeBlocks / 2; ++i)
        raw[i].load(row + (size_t)min(b0 + 2 * i, nb - 1) * Quarter<TYPE>::kBlockBytes, g);
    uint8_t* const base = out + (size_t)tile * nb * (4 * kSlabTileBytes);
#pragma unroll
    for (uint32_t i = 0; i < kDecodeBlocks / 2; ++i) {
        PackedOperands<DT> packed;
        raw[i].decode_into(g, packed);
        if (i > 0) __syncthreads();   // the images have been read
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const uint32_t k = Quarter<TYPE>::klocal(g, s), step = ((k >> 4) & 2u) | ((k >> 3) & 1u);
            *reinterpret_cast<uint4*>(&image[wave >> 1][(k >> 6) * kSlabTileBytes + step * 1024 + ((k >> 4) & 1u) * 512 + column * 16]) =
                packed.operand(s);
        }
        __syncthreads();
        const uint32_t b = b0 + 2 * i;
        if (b < nb) {   // a wave stores half of its super-block's image
            const uint32_t at = (wave & 1u) * 8192 + lane * 16;
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j)
                *reinterpret_cast<uint4*>(base + (size_t)b * (4 * kSlabTileBytes) + at + 1024 * j) =
                    *reinterpret_cast<const uint4*>(&image[wave >> 1][at + 1024 * j]);
        }
    }
}

template <int DT>
__device__ __forceinline__ float16v mfma32(uint4 a, uint4 b, float16v c) {
    if constexpr (DT == 1) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
}

// cache bits of a buffer access that is coherent across the chip's L2 slices, as a relaxed atomic of device scope is: sc1
constexpr int kDeviceScope = 16;

struct DecodedParams {
    const uint8_t* panel;
    const uint16_t* x;
    void* y;
    uint32_t m, n, nb, y_dtype;   // n: the matrix's columns (the stride of y)
    uint32_t first, columns;      // the panel's
    uint32_t tiles_m, tiles_n;
    // K in two segments:
    uint8_t* sums;                // [tile][wave][32 x 32 tile][element / 4][lane], of whichever segment of a tile ends first
    uint32_t* counters;           // [tile][1 + waves], zero between launches
};

// as many stages as fit 160 KB
constexpr uint32_t stages_of(uint32_t stage_bytes) { return std::min(5u, 163840u / stage_bytes); }

// A workgroup is eight waves, 8 / WN x WN along rows and columns; a wave multiplies 32 RT rows by 32 NT columns.  32 K of all
// rows and columns of the tile are a stage, and four or five stages a ring in LDS: one is multiplied, the next has landed,
// the others are on their way.  Two multiplying waves a SIMD: one hides the other's reads and scalar instructions (four waves
// of 128 x 128 with half the fragment reads take 157 us for the 142 below, four of 64 x 160 32 ns a multiplication).
// Measured at 2048 x 8192 x 5120 (256 tiles of 256 x 256, one round): 142 us = 1.21 PFLOP/s; on zeros, where the chip keeps
// its clock, 117, of which the stores are 12 and waiting for loads 13 (26 with two stages of 64 K); the matrix instruction
// alone takes 95 us on random operands.
template <int DT, int RT, int NT, int WN, bool CUT, bool FOURS>
__global__ __launch_bounds__(512) void gemm_decoded_kernel(const DecodedParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    constexpr uint32_t kWaves = 8, kWavesM = kWaves / WN;
    constexpr uint32_t kRows = kWavesM * 32 * RT, kColumnTiles = WN * NT;
    constexpr uint32_t kRowsStage = kRows * 64, kStage = kRowsStage + kColumnTiles * 2048;
    constexpr uint32_t kStages = stages_of(kStage);
    constexpr int kRowLoads = (int)(kRowsStage / 1024 / kWaves), kColumnLoads = (int)((kColumnTiles * 2 + kWaves - 1) / kWaves);
    constexpr int kLoads = kRowLoads + kColumnLoads, kFrags = RT + NT, kMul = RT * NT;
    static_assert(kRowsStage % (1024 * kWaves) == 0, "whole instructions per wave");

    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t wave_m = wave / WN, wave_n = wave % WN;
    uint32_t tile, tile_m, tile_n, segment;
    {   // XCD x takes the x-th eighth of the (column tile, row tile, segment) list: the row tiles of a column tile share it in an L2
        const uint32_t items = p.tiles_m * p.tiles_n * (CUT ? 2u : 1u), xcd = blockIdx.x & 7u, at = blockIdx.x >> 3;
        const uint32_t begin = (uint32_t)((uint64_t)items * xcd >> 3), end = (uint32_t)((uint64_t)items * (xcd + 1) >> 3);
        if (begin + at >= end) return;
        tile = CUT ? (begin + at) >> 1 : begin + at;
        segment = CUT ? (begin + at) & 1u : 0u;
        tile_n = tile / p.tiles_m;
        tile_m = tile - tile_n * p.tiles_m;
    }
    const uint32_t m0 = tile_m * kRows, k = p.nb << 8, all_halves = p.nb * 8;   // 32 K each
    const uint32_t first_half = segment * (p.nb / 2) * 8;
    const uint32_t halves = !CUT ? all_halves : segment ? all_halves - first_half : p.nb / 2 * 8;
    const uint32_t r32 = lane & 31u, kg = lane >> 5;

    float16v acc[RT][NT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    // Rows: a load instruction brings 16 rows; the 16-byte piece q of row r sits at unit 4 r + (q ^ ((r >> 2) & 3)), which
    // spreads the rows a fragment read touches over all banks.  Instruction i of a wave is piece 8 i + wave.  (rows past m
    // are clamped: they only feed outputs that are never stored)
    uint32_t row_offset[kRowLoads];
#pragma unroll
    for (int i = 0; i < kRowLoads; ++i) {
        const uint32_t r = 16 * ((uint32_t)i * kWaves + wave) + (lane >> 2);
        row_offset[i] = (min(m0 + r, p.m - 1) - m0) * k * 2 + 16 * ((lane & 3u) ^ ((r >> 2) & 3u));
    }
    const uint8_t* rows = reinterpret_cast<const uint8_t*>(p.x + (size_t)m0 * k) + (size_t)first_half * 64;
    // Columns: two kilobyte steps of each of the tile's 32-column tiles (past the panel its last one again; pieces past the
    // tile repeat its first ones, the same bytes to the same place, so that all waves count the same loads)
    const uint32_t last_tile = (p.columns + 31) / 32 - 1;
    uint32_t column_offset[kColumnLoads], column_to[kColumnLoads];
#pragma unroll
    for (int i = 0; i < kColumnLoads; ++i) {
        const uint32_t piece = ((uint32_t)i * kWaves + wave) % (2 * kColumnTiles);
        column_offset[i] = (min(tile_n * kColumnTiles + (piece >> 1), last_tile) - tile_n * kColumnTiles) * (all_halves / 2) * kSlabTileBytes +
                           1024 * (piece & 1u) + 16 * lane;
        column_to[i] = kRowsStage + 1024 * piece;
    }
    const uint8_t* columns = p.panel + (size_t)tile_n * kColumnTiles * (all_halves / 2) * kSlabTileBytes + (size_t)first_half * 2048;
    const uint32_t lds_at = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)lds);
    auto load = [&](uint32_t half, uint32_t stage, int i) {
        const uint32_t to = lds_at + stage * kStage;
        if (i < kRowLoads) lds_load16_at(rows + (size_t)half * 64, row_offset[i], to + 1024 * (kWaves * i + wave));
        else lds_load16_at(columns + (size_t)half * 2048, column_offset[i - kRowLoads], to + column_to[i - kRowLoads]);
    };
    const uint32_t sw = (r32 >> 2) & 3u;
    const uint32_t a_even = wave_m * (32 * RT * 64) + (4 * r32 + ((2 * kg) ^ sw)) * 16;
    const uint32_t a_odd = wave_m * (32 * RT * 64) + (4 * r32 + ((2 * kg + 1) ^ sw)) * 16;
    const uint32_t b_at = kRowsStage + wave_n * NT * 2048 + 16 * lane;
    struct Frags {
        uint4 v[kFrags];
    };
    auto read = [&](Frags& f, uint32_t stage, int s, int t) {
        const uint8_t* const from = lds + stage * kStage;
        f.v[t] = t < RT ? *reinterpret_cast<const uint4*>(from + (s ? a_odd : a_even) + t * 2048)
                        : *reinterpret_cast<const uint4*>(from + b_at + (t - RT) * 2048 + s * 1024);
    };
    // One step: the multiplications of `cur`; between them, one at a time so that each hides behind a multiplication in
    // flight, the reads of step `s` of `stage` into `next` and the load instructions of `half` into stage `into`.
    auto step = [&](const Frags& cur, Frags& next, uint32_t stage, int s, auto with_reads, auto with_loads, uint32_t half, uint32_t into) {
        constexpr int kSlots = std::max(kMul, std::max(kFrags, kLoads));
#pragma unroll
        for (int idx = 0; idx < kSlots; ++idx) {
            if constexpr (decltype(with_reads)::value)
                if (idx < kFrags) read(next, stage, s, idx);
            if constexpr (decltype(with_loads)::value)
                if (idx >= kSlots - kLoads) load(half, into, idx - (kSlots - kLoads));
            if (idx < kMul) {
                const uint4 row = cur.v[idx % RT], column = cur.v[RT + idx / RT];
                acc[idx % RT][idx / RT] = mfma32<DT>(FOURS ? column : row, FOURS ? row : column, acc[idx % RT][idx / RT]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};

    Frags f0, f1;
#pragma unroll
    for (uint32_t h = 0; h < kStages - 1; ++h)   // (at least eight half slabs)
#pragma unroll
        for (int i = 0; i < kLoads; ++i) load(h, h, i);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kStages - 2) * kLoads) : "memory");
    __syncthreads();
#pragma unroll
    for (int t = 0; t < kFrags; ++t) read(f0, 0, 0, t);
    // Software pipeline, one step deep: the fragments of a step are read while the one before multiplies, also across the
    // barrier that opens a stage.
    uint32_t stage = 0, into = kStages - 1;
    for (uint32_t c = 0; c + 1 < halves; ++c) {
        const uint32_t next = stage == kStages - 1 ? 0 : stage + 1;
        // into the stage that the last barrier freed (past the end the last half slab again, where nothing reads any more)
        step(f0, f1, stage, 1, yes, yes, min(c + kStages - 1, halves - 1), into);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kStages - 2) * kLoads) : "memory");   // half slab c + 1 has landed
        __syncthreads();   // in every wave; and this one's fragments are all in registers
        __builtin_amdgcn_sched_barrier(0);
        step(f1, f0, next, 0, yes, no, 0u, 0u);
        into = stage;
        stage = next;
    }
    step(f0, f1, stage, 1, yes, no, 0u, 0u);
    step(f1, f0, stage, 0, no, no, 0u, 0u);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the spare loads

    // K in two segments: the one that ends first leaves its sums in the scratch, the other adds them to its own (of two the
    // order does not matter) and stores.  The first waits for nothing, the other for stores that are already under way, wave
    // by wave.  Device-scope accesses: coherent across the chip's L2 slices without cache-wide flushes.
    constexpr uint32_t kSumBytes = kMul * 4096;   // of a wave
    __amdgpu_buffer_rsrc_t sums;
    if constexpr (CUT) {
        uint32_t* const counters = p.counters + (size_t)tile * (1 + kWaves);
        uint32_t* const ready = counters + 1 + wave;
        sums = __builtin_amdgcn_make_buffer_rsrc(
            reinterpret_cast<void*>(uniform_address(p.sums + ((size_t)tile * kWaves + wave) * kSumBytes)), 0, kSumBytes, 0x00027000);
        __syncthreads();   // the last stages have been read
        if (tid == 0)
            *reinterpret_cast<uint32_t*>(lds) = __hip_atomic_fetch_add(counters, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        const uint32_t place = (uint32_t)__builtin_amdgcn_readfirstlane((int)*reinterpret_cast<const uint32_t*>(lds));
        if (place == 0) {
#pragma unroll
            for (int i = 0; i < kMul; ++i) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float16v& c = acc[i % RT][i / RT];
                    const u32x4 part = {__float_as_uint(c[4 * q]), __float_as_uint(c[4 * q + 1]), __float_as_uint(c[4 * q + 2]),
                                        __float_as_uint(c[4 * q + 3])};
                    __builtin_amdgcn_raw_buffer_store_b128(part, sums, 16 * lane, 4096 * i + 1024 * q, kDeviceScope);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): they have completed
            if (lane == 0) __hip_atomic_store(ready, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
        while (__hip_atomic_load(ready, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) __builtin_amdgcn_s_sleep(8);
        asm volatile("" ::: "memory");
        if (lane == 0) __hip_atomic_store(ready, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (tid == 0) __hip_atomic_store(counters, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // FOURS, an output whose rows are whole fours: the columns are the instruction's rows, and elements 4 q .. 4 q + 3 of a lane
    // are columns 8 q + 4 kg .. of row r32.  Else the rows are, the elements rows 8 q + 4 kg .. of column r32, and lanes store
    // along a row.
    auto store = [&](auto type) {
        constexpr uint32_t kType = decltype(type)::value;
#pragma unroll
        for (int i = 0; i < RT; ++i) {
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const uint32_t row0 = m0 + 32 * (wave_m * RT + i), column0 = 32 * (tile_n * kColumnTiles + wave_n * NT + j);
                u32x4 part[4];
                if constexpr (CUT) {
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        part[q] = __builtin_amdgcn_raw_buffer_load_b128(sums, 16 * lane, 4096 * (j * RT + i) + 1024 * q, kDeviceScope);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = CUT ? acc[i][j][4 * q + e] + __uint_as_float(part[q][e]) : acc[i][j][4 * q + e];
                    if constexpr (FOURS) {   // (a panel's columns come in fours, too)
                        const uint32_t row = row0 + r32, column = column0 + 8 * q + 4 * kg;
                        if (row >= p.m || column >= p.columns) continue;
                        const size_t at = (size_t)row * p.n + p.first + column;
                        if constexpr (kType == FH_F32)
                            *reinterpret_cast<float4*>(static_cast<float*>(p.y) + at) = make_float4(v[0], v[1], v[2], v[3]);
                        else if constexpr (kType == FH_F16)
                            *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.y) + at) =
                                make_uint2(f32_to_f16_bits(v[0]) | (f32_to_f16_bits(v[1]) << 16),
                                           f32_to_f16_bits(v[2]) | (f32_to_f16_bits(v[3]) << 16));
                        else
                            *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p.y) + at) =
                                make_uint2(f32_pair_to_bf16_bits(v[0], v[1]), f32_pair_to_bf16_bits(v[2], v[3]));
                    } else {
                        const uint32_t column = column0 + r32;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const uint32_t row = row0 + 8 * q + 4 * kg + e;
                            if (row < p.m && column < p.columns)
                                store_from_f32(p.y, (size_t)row * p.n + p.first + column, kType, v[e]);
                        }
                    }
                }
                if constexpr (CUT) __builtin_amdgcn_sched_barrier(0);   // (the sums of another tile do not fit the registers)
            }
        }
    };
    if (p.y_dtype == FH_F32) store(std::integral_constant<uint32_t, FH_F32>{});
    else if (p.y_dtype == FH_F16) store(std::integral_constant<uint32_t, FH_F16>{});
    else store(std::integral_constant<uint32_t, FH_BF16>{});
}

template <int DT, int RT, int NT, int WN, bool CUT, bool FOURS>
void launch_product(hipStream_t s, DecodedParams p) {
    constexpr uint32_t kRows = 8 / WN * 32 * RT, kColumns = WN * NT * 32;
    constexpr uint32_t kStage = kRows * 64 + kColumns * 64;
    constexpr size_t kLds = kStage * stages_of(kStage);
    static std::atomic<uint64_t> raised{0};
    once_per_device(raised, [] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_decoded_kernel<DT, RT, NT, WN, CUT, FOURS>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds);
    });
    p.tiles_m = (p.m + kRows - 1) / kRows;
    p.tiles_n = (p.columns + kColumns - 1) / kColumns;
    const uint32_t items = p.tiles_m * p.tiles_n * (CUT ? 2u : 1u);
    hipLaunchKernelGGL((gemm_decoded_kernel<DT, RT, NT, WN, CUT, FOURS>), dim3((items + 7) / 8 * 8), dim3(512), kLds, s, p);
}

template <int DT>
void launch_decode(hipStream_t s, uint32_t ggml_type, const uint8_t* w, uint8_t* out, uint32_t columns, uint32_t nb) {
    const dim3 grid((nb + kDecodeBlocks - 1) / kDecodeBlocks, (columns + 31) / 32);
    switch (ggml_type) {
        case kQ4K: hipLaunchKernelGGL((decode_panel_kernel<kQ4K, DT>), grid, dim3(256), 0, s, w, out, columns, nb); break;
        case kQ5K: hipLaunchKernelGGL((decode_panel_kernel<kQ5K, DT>), grid, dim3(256), 0, s, w, out, columns, nb); break;
        case kQ6K: hipLaunchKernelGGL((decode_panel_kernel<kQ6K, DT>), grid, dim3(256), 0, s, w, out, columns, nb); break;
        case kIQ4XS: hipLaunchKernelGGL((decode_panel_kernel<kIQ4XS, DT>), grid, dim3(256), 0, s, w, out, columns, nb); break;
        default: hipLaunchKernelGGL((decode_panel_kernel<kQ8_0, DT>), grid, dim3(256), 0, s, w, out, columns, nb); break;
    }
}

template <int DT, bool CUT, bool FOURS>
void launch_tile(hipStream_t s, const DecodedParams& p, uint32_t columns) {
    if (columns == 192) launch_product<DT, 2, 3, 2, CUT, FOURS>(s, p);
    else if (columns == 320) launch_product<DT, 2, 5, 2, CUT, FOURS>(s, p);
    else launch_product<DT, 4, 2, 4, CUT, FOURS>(s, p);
}

// Four outputs of a row in a store of a lane take 694 us where single ones of neighbouring columns take 706 (1999 x 34816 x 5120, 320
// columns; 8192 x 4096, 1500 rows, 256 columns asked for: 115 / 119), but only where every row starts on a four.
template <int DT>
void launch_tile_of(hipStream_t s, const DecodedParams& p, uint32_t columns, bool cut) {
    if (p.n % 4 == 0) cut ? launch_tile<DT, true, true>(s, p, columns) : launch_tile<DT, false, true>(s, p, columns);
    else cut ? launch_tile<DT, true, false>(s, p, columns) : launch_tile<DT, false, false>(s, p, columns);
}

// What a round of 256 workgroups of a tile takes, in us: a start (first loads, stores) and a time per 5120 of K (rows of real
// data, where the chip lowers its clock; of zeros a round of 256 x 256 takes a sixth less).
struct DecodedTile {
    uint32_t columns;
    double start, round;
};
constexpr DecodedTile kDecodedTiles[] = {{192, 9.2, 101.2}, {256, 11.6, 121.2}, {320, 13.5, 149.6}};
constexpr size_t kMostPanelBytes = fh_device::kScratchOptional;
constexpr double kDecodeUs = 3.8;      // of every panel
constexpr double kRunUs = 5.0;         // and of every run of tiles behind the first
constexpr double kExchangeUs = 1.64;   // per million outputs whose two segments meet in memory

double rounds_us(const DecodedTile& t, double rounds, uint32_t k) {
    const double whole = (double)(uint64_t)rounds, part = rounds - whole;
    return t.start * (whole + (part > 0)) + (whole + (part > 0 ? 0.54 + 0.46 * part : 0.0)) * t.round * k / 5120.0;
}

// A run of column tiles in panels that fit the scratch, each but the last of as many tiles as make whole rounds; 0 where not
// even one tile fits.
double run_us(const DecodedTile& t, uint32_t columns, uint32_t tiles_m, uint32_t k, uint32_t cus, uint32_t* panel) {
    const uint64_t most = kMostPanelBytes / ((uint64_t)k * 2 * t.columns);
    if (most == 0) return 0.0;
    const uint32_t tiles_n = (columns + t.columns - 1) / t.columns;
    uint32_t tiles = (uint32_t)std::min<uint64_t>(most, tiles_n);
    if (tiles < tiles_n && (uint64_t)tiles * tiles_m > cus)
        tiles = std::max(1u, (uint32_t)((uint64_t)tiles * tiles_m / cus * cus / tiles_m));
    double us = 0.0;
    for (uint32_t first = 0; first < tiles_n; first += tiles)
        us += kDecodeUs + rounds_us(t, (double)std::min(tiles, tiles_n - first) * tiles_m / cus, k);
    *panel = tiles * t.columns;
    return us;
}

}  // namespace

// The decode by its bytes, then rounds of the product, the last one cheaper where it is not full; against the fused tiles'
// estimate.  Of the 500 products of 400 - 2048 rows and K of 512 - 17408 in profiles/decoded_runs_us.txt, none of which the constants
// were fitted to, 236 decode, three of them slower than the fused tiles by more than 2%, and the dispatched time is 1.9% from the fastest
// in the mean.  264 stay fused; 50 of those lose more than 5% by it and 24 more than 10%, where the fused estimate is too
// low (Q6_K 411 x 21004 x 6144 272 against 217 us).
//
// Runs of tiles.  A round of a tile takes what it takes however few workgroups it has, so columns that do not make whole rounds of
// one tile are better cut into whole rounds of one and the rest on another: 1999 x 34816 x 5120 is 3.4 rounds of 320 columns, 717 us, or
// one of those and three of 256 columns, 687 (three of 30,000 random products would gain by a third tile).  All tiles sum in the same order.
//
// Two segments of K.  5120 columns and 1999 rows are 128 tiles of 320 x 256: half of the chip, or 216 of 192 columns.  Cut in two, the
// former are one round.  Q6_K 1999 x 5120 x 17408 uncut 401 (192 columns), 456 (320), cut 349 us (320), fused tiles 421; Q4_K 392 / 450
// / 343 / 353; 1999 x 5120 x 5120 stays uncut, 114 / 125 / 122 / 118.
//
// us, fused tiles / 192 / 256 / 320 columns: Q4_K 1999 x 34816 x 5120 775 / 777 / 745 / 717; 1500 x 8192 x 4096 127 / 162 / 111 / 116 (it
// stays fused, whose estimate is lower); Q8_0 2048 x 4096 x 4096 100 / 83 / 85 / 98.
bool gemm_takes_decoded(GemmArgs& a) {
    if (a.decoded_min_rows == 0 || a.wide32_tile != 0 || a.wide_shape != 1 || !a.resident_switch || a.m <= 256) return false;
    const uint32_t cus = a.cu_count > 0 ? (uint32_t)a.cu_count : 256u, tiles_m = (a.m + 255) / 256;
    const bool forced = a.decoded_min_rows > 1;   // from that many rows on, whatever the estimates say
    if (forced && a.m < (uint32_t)a.decoded_min_rows) return false;
    // (Q6_K's fused estimate is 2 - 4% high from 512 rows on: 768 x 28672 x 4096 245 us there, 271 here; a product that only the square
    // tiles take, few columns and rows too long to be resident, has none: 300 x 512 x 4096 36 us there, 71 to 101 here)
    // Rows of one super-block are all starts and stores, which the fused estimate puts too high: 786 x 144422 x 256 Q5_K 178 us
    // there, 228 here, nine of eleven such products slower (profiles/routes_us.txt); from two super-blocks on they gain.
    const double fused = forced ? 1e300 : gemm_fused_estimate(a);
    if (!forced && (fused >= 1e300 || a.k < 512)) return false;
    double best = a.ggml_type == kQ6K ? 0.96 * fused : fused;
    DecodedPlan& plan = a.decoded;
    const double decode = (double)a.n * a.k * (2.0 + block_bytes(a.ggml_type) / 256.0) / 4.69e6;
    const bool any_tile = a.decoded_tile == 0;
    // whole rounds of one tile and the rest on another: a round takes what its tile does, however few of its workgroups there are
    for (const DecodedTile& last : kDecodedTiles) {
        if (!any_tile && (uint32_t)a.decoded_tile != last.columns) continue;
        for (const DecodedTile& one : kDecodedTiles) {
            const uint32_t one_round = cus / tiles_m * one.columns, one_most = any_tile && &one != &last ? (a.n - 1) / std::max(one_round, 1u) : 0u;
            for (uint32_t i = 0; i <= (one_round ? one_most : 0u); ++i) {
                if (i == 0 && &one != kDecodedTiles) continue;   // (the same plan from every tile)
                DecodedPlan p{};
                double us = decode;
                auto add = [&](const DecodedTile& t, uint32_t columns) {
                    DecodedPlan::Run& run = p.run[p.runs++];
                    run.columns = columns;
                    run.tile = t.columns;
                    const double here = run_us(t, columns, tiles_m, a.k, cus, &run.panel);
                    us += here == 0.0 ? 1e300 : here + (p.runs > 1 ? kRunUs : 0.0);
                };
                if (i > 0) add(one, i * one_round);
                add(last, a.n - i * one_round);
                if (us < best) {
                    best = us;
                    plan = p;
                    plan.segments = 1;
                }
            }
        }
    }
    for (int i = 0; i < plan.runs; ++i)
        plan.panel_bytes = std::max(plan.panel_bytes, (size_t)(std::min(plan.run[i].panel, plan.run[i].columns) + 31) / 32 * 32 * a.k * 2);
    // Two segments of K: one panel, whose tiles come twice with half of the length
    if (a.decoded_segments == 2 || (a.decoded_segments == 0 && !forced)) {
        if (a.decoded_segments == 2) best = 1e300;
        for (const DecodedTile& t : kDecodedTiles) {
            if ((!any_tile && (uint32_t)a.decoded_tile != t.columns) || a.k < 512) continue;
            const uint64_t tiles = (uint64_t)((a.n + t.columns - 1) / t.columns) * tiles_m;
            const size_t panel_bytes = (size_t)(a.n + 31) / 32 * 32 * a.k * 2, sum_bytes = tiles * 256 * t.columns * 4;
            if (panel_bytes + sum_bytes > kMostPanelBytes || tiles * 9 > fh_device::kCounterWords) continue;
            const double us = decode + kDecodeUs + kExchangeUs * 1e-6 * a.m * a.n + rounds_us(t, 2.0 * (double)tiles / cus, a.k / 2);
            if (us < best) {
                best = us;
                plan = DecodedPlan{};
                plan.run[0] = {a.n, t.columns, a.n};
                plan.runs = 1;
                plan.segments = 2;
                plan.panel_bytes = panel_bytes;
                plan.sum_bytes = sum_bytes;
            }
        }
    }
    return plan.runs != 0;
}

void launch_gemm_decoded(hipStream_t s, const GemmArgs& a) {
    const uint32_t nb = a.k / 256;
    const DecodedPlan& plan = a.decoded;
    DecodedParams p{};
    uint8_t* const out = reinterpret_cast<uint8_t*>(a.partials);
    p.panel = out;
    p.x = static_cast<const uint16_t*>(a.x);
    p.y = a.y;
    p.m = a.m;
    p.n = a.n;
    p.nb = nb;
    p.y_dtype = a.y_dtype;
    p.sums = out + plan.panel_bytes;
    p.counters = a.counters;
    const size_t row_bytes = (size_t)nb * block_bytes(a.ggml_type);
    uint32_t first = 0;
    for (int i = 0; i < plan.runs; ++i) {
        const DecodedPlan::Run& run = plan.run[i];
        const uint32_t end = first + run.columns;
        for (; first < end; first += p.columns) {
            p.first = first;
            p.columns = std::min(run.panel, end - first);
            const uint8_t* const w = static_cast<const uint8_t*>(a.w) + first * row_bytes;
            if (a.x_dtype == FH_F16) {
                launch_decode<1>(s, a.ggml_type, w, out, p.columns, nb);
                launch_tile_of<1>(s, p, run.tile, plan.segments == 2);
            } else {
                launch_decode<2>(s, a.ggml_type, w, out, p.columns, nb);
                launch_tile_of<2>(s, p, run.tile, plan.segments == 2);
            }
        }
    }
}

}  // namespace fh
