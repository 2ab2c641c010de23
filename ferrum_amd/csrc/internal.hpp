// Shared definitions of the gfx950 backend: device objects, error plumbing and
// the host-side launchers each kernel file exports.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <cstdio>
#include <utility>
#include <vector>
#include <string>

#include "../../include/ferrum_hip.h"
#include "../../include/ferrum_hip_probe.h"
#include "freed_blocks.hpp"

// Kernel-selection switches, set by name through fh_set_tuning (kTuningKeys in capi.hip).
struct fh_tuning {
    int64_t k_quant_gemv_ksplit = 0;   // 0 = automatic
    int64_t gemm_min_rows = 2;         // smallest M that takes the MFMA tile path
    int64_t gemm_wide_shape = 1;       // matrix instruction of the 128- and 256-row tiles: 0 = 16x16x32, 1 = whichever is estimated faster, 2 = 32x32x16
    int64_t gemm_wide32_tile = 0;      // 0 = by shape; 12, 14, 15 (128-row tile x 64, 128, 160 columns), 24, 25 (256-row tile)
    int64_t gemm_wide32_segments = 0;  // K segments of the 32x32x16 form: 0 = by shape (a forced tile or form: uncut), else at most that many, up to 8 (a forced tile: exactly)
    int64_t gemm_decoded_min_rows = 1; // products that decode their weights into the scratch first: 0 never, 1 where estimated faster, else from that many rows on (and 257), fewer never
    int64_t gemm_decoded_tile = 0;     // their tile: 0 = by shape; 192, 256 or 320 columns
    int64_t gemm_decoded_segments = 0; // and their K segments: 0 = by shape, 1 = uncut, 2 = two
    int64_t gemm_wide_min_rows = 33;   // smallest M that takes the 256-row tile (it wins from there up)
    int64_t gemm_skinny_max_rows = 64; // with gemm_resident 0: largest M that takes the few-rows kernel (0 = never)
    int64_t expert_grouped_min_assignments = 32;  // fewest assignments grouped by expert (0 = never)
    int64_t moe_fold_route = 1;        // fh_moe_ffn, one token: the gate|up launch routes the token itself (0 = a moe_route launch first)
    int64_t gemm_few_tiles_split = 1;  // few rows: a tile's super-blocks dealt over the waves, any K: 0 never (whole tiles per wave, the kernels for rows that fit LDS or not), 1 where it wins, 2 wherever it runs
    int64_t moe_fold_combine = 1;      // fh_moe_ffn with few tokens: down projection and weighted sum in one launch (0 = two)
    int64_t gemm_resident = 1;         // rows that fit LDS whole take the rows-resident kernel (0 = square tiles)
    int64_t gemv_ring = 1;   // streamed GEMVs of one row keep a workgroup on every compute unit: 1 where that is faster, 0 never, 2 wherever it fits
    int64_t gemv_stream_own_loads = 1; // the streamed Q4_K GEMV's waves load the super-blocks they multiply (tiles of up to 14 rows); 0: the tile row by row
    int64_t expert_weight_ring = 1;    // grouped Q4_K / Q6_K expert projection with short rows: weights through LDS rings (0 = straight into registers)
    int64_t gemv_stream = 1;           // dense Q4_K / Q6_K GEMV on the streamed matrix-core kernel: 0 never, 1 where it wins, 2 wherever it runs
    int64_t moe_routing_temporary_limit = 128ll << 20;  // bytes of routing temporaries per SparseMoe chunk (src/metal/legacy.rs:95)
    int64_t gemm_f32_min_rows = 0;     // f32 activations take the f16 tile kernels from this many rows (0 = never)
    int64_t allocation_limit_bytes = 0;  // requests for more fail as on a GPU without room (0 = none)
    int64_t probe_read_form = 0;       // fh_probe_read: 100 x threads per workgroup + loads per lane (+ 1000000: LDS-direct loads); 0 = 256 x 8
};

struct fh_device {
    // The device object lives until fh_device_destroy has been called and the last buffer,
    // matrix, graph or event created on it is gone: their release functions read it.
    std::atomic<int> handles{1};   // the caller's own handle, plus one per live object
    bool closed = false;   // fh_device_destroy has run: the stream is gone, memory is freed directly
    int ordinal = 0;
    hipStream_t stream = nullptr;
    hipDeviceProp_t props{};
    const char* last_operation = "";
    int64_t last_rows_plan = 0;   // of the last dense product: 0, or the few-rows kernel's rows, tiles and K segments
    int64_t last_decoded_tile = 0;   // ... and 0, or the columns of its (first) tile where its weights were decoded first
    int64_t last_decoded_cut = 0;    // ... where its K was cut in two besides: this one and not the one before
    int64_t last_decoded_runs = 0;   // ... and its runs of tiles
    std::atomic<bool> capturing{false};   // set under freed.settling: what empties the pool waits on the stream
    fh_tuning tuning;
    // Blocks of freed buffers, by size, for the buffers to come (fh_buffer_alloc): hipMalloc and hipFree
    // take 10 - 20 us each and the latter waits for the GPU (a routed FFN of 200 f32 tokens whose operators
    // return new tensors: 453 us without the pool, 286 with it).  All work of the library on a buffer is on
    // `stream`, so a block can be handed on at once.  What has been done elsewhere with a buffer whose address has left the
    // library only a wait for the whole GPU covers: such blocks gather, and one wait serves all of them (the same FFN, three
    // of its outputs seen by torch: a wait for each, 110 us of host time, kept the host from running ahead: 248 us, now 205).
    // Python may drop a buffer on any thread, and another device object on the same GPU that finds no memory
    // empties this one's pool: the pool has a lock.
    fh::FreedBlocks freed;
    fh_device* next_live = nullptr;   // device objects that have not been destroyed (g_live in capi.hip)
    // scratch owned by the device: [counter words | floats / ids]
    void* scratch = nullptr;
    size_t scratch_bytes = 0;
    // this device's copy of the library's fixed scratch array (fh_project_quantized_no_alloc)
    void* fixed_scratch = nullptr;
    static constexpr size_t kCounterWords = 1u << 16;
    static constexpr size_t kScratchFloor = 16u << 20;   // the data area is never smaller
    static constexpr size_t kScratchOptional = 256u << 20;   // nor grown beyond this by kernels that only save time by it
    size_t scratch_refused = 0;      // bytes such a kernel asked for in vain (0 = none)
    uint32_t scratch_wait = 0;       // calls that take it for refused before the next request
    // Releases asked for while an execution is being recorded wait for its end:
    // freeing or synchronizing inside a stream capture would invalidate it.
    // scratch blocks that were outgrown while recorded executions (which carry their address)
    // were alive: freed with the last of those
    std::vector<void*> retired_scratch;
    // temporaries of fh_moe_ffn: one block, grown like the scratch and retired with it
    fh_buffer* workspace = nullptr;
    // activations rewritten to the width of a matrix whose rows are stored padded: grown the same way
    fh_buffer* padded_rows = nullptr;
    int live_graphs = 0;
    std::vector<void*> deferred_frees;
    std::vector<std::pair<hipGraphExec_t, hipGraph_t>> deferred_graphs;
};

struct fh_buffer {
    fh_device* device = nullptr;
    void* ptr = nullptr;
    size_t bytes = 0;
    size_t capacity = 0;    // bytes of the block behind ptr
    bool exposed = false;   // fh_buffer_device_ptr has handed out the address
};

struct fh_qmatrix {
    fh_device* device = nullptr;
    void* ptr = nullptr;
    size_t bytes = 0;
    uint32_t ggml_type = 0;
    uint64_t rows = 0;     // per expert
    uint64_t cols = 0;
    uint64_t experts = 1;
    // Width of a stored row, a multiple of 256: `cols` except for a Q8_0 matrix whose rows are 32 n
    // weights with n not a multiple of 8, which is kept with every row padded by empty blocks
    // (scale and quants zero) so that the kernels see runs of eight blocks.
    uint64_t stored_cols = 0;
    bool padded() const { return stored_cols != cols; }
};

struct fh_graph {
    fh_device* device = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
};

struct fh_event {
    fh_device* device = nullptr;
    hipEvent_t event = nullptr;
};

namespace fh {

fh_status fail(fh_status code, const char* fmt, ...);
fh_status hip_fail(hipError_t err, const char* what);

constexpr uint32_t kQ4K = FH_GGML_Q4_K;
constexpr uint32_t kQ5K = FH_GGML_Q5_K;
constexpr uint32_t kQ6K = FH_GGML_Q6_K;
constexpr uint32_t kIQ4XS = FH_GGML_IQ4_XS;
constexpr uint32_t kQ8_0 = FH_GGML_Q8_0;

// bytes of 256 weights: one super-block, or eight 34-byte blocks of Q8_0
constexpr uint32_t block_bytes_of(uint32_t ggml_type) {
    return ggml_type == kQ4K     ? 144u
           : ggml_type == kQ5K   ? 176u
           : ggml_type == kQ6K   ? 210u
           : ggml_type == kIQ4XS ? 136u
           : ggml_type == kQ8_0  ? 272u
                                 : 0u;
}

inline size_t block_bytes(uint32_t ggml_type) {
    return block_bytes_of(ggml_type);
}
// Runs `raise` once for the current device (two threads may both, on ordinals from 64 on every call does): a
// kernel's dynamic LDS limit belongs to its copy on a device.
template <class Raise>
void once_per_device(std::atomic<uint64_t>& done, Raise&& raise) {
    int ordinal = 64;
    (void)hipGetDevice(&ordinal);
    const uint64_t bit = ordinal < 64 ? 1ull << ordinal : 0;
    if ((done.load(std::memory_order_acquire) & bit) != 0) return;
    raise();
    done.fetch_or(bit, std::memory_order_release);
}

inline size_t dtype_bytes(uint32_t dtype) { return dtype == FH_F32 ? 4 : 2; }

// ---- launchers (one per kernel family); each returns the kernel name ----

// dequant.hip
// f32 -> f16 (round to nearest even), `count` a multiple of 8: activations on their way to the tile kernels
// scratch the search needs for maxima of pieces of a row (plus a counter word per row); 0: none
size_t argmax_partial_bytes(uint32_t rows, uint32_t width);
const char* launch_argmax_rows(hipStream_t s, const void* logits, uint32_t dtype, uint32_t rows, uint32_t width,
                               void* partial, uint32_t* counters, uint32_t* out);
void launch_round_to_f16(hipStream_t s, const float* in, uint16_t* out, size_t count);
// rows are stored `cols` wide (a multiple of 256) and written `out_cols` wide
const char* launch_dequantize(hipStream_t s, uint32_t ggml_type, const void* w, size_t rows,
                              size_t cols, size_t out_cols, void* out, uint32_t out_dtype);
// pieces of `cols` elements (a multiple of 32) -> pieces of `padded` elements, zero beyond `cols`
void launch_pad_rows(hipStream_t s, const void* in, void* out, size_t pieces, size_t cols, size_t padded,
                     size_t element_bytes);
const char* launch_embedding_gather(hipStream_t s, uint32_t ggml_type, const void* w, size_t cols, size_t out_cols,
                                    const uint32_t* ids_dev, size_t count, void* out,
                                    uint32_t out_dtype);

// probe.hip: measurement kernels (a plain 128-bit read of a buffer; an MFMA issue loop)
const char* launch_read_probe(hipStream_t s, const void* data, size_t bytes, uint32_t* sink, int64_t form);
const char* launch_mfma_probe(hipStream_t s, int shape, uint32_t groups, uint32_t iterations, float* sink,
                              double* flops);
const char* launch_coissue_probe(hipStream_t s, uint32_t groups, uint32_t iterations, uint32_t mfma,
                                 uint32_t valu_rounds, float* sink);

// norm.hip
// residual = round(a + b), normed = rmsnorm(residual) * weight; all operands of one dtype,
// no output overlapping an operand or the other output.
const char* launch_add_rmsnorm(hipStream_t s, const void* a, const void* b, const void* weight, void* residual,
                               void* normed, uint32_t rows, uint32_t width, uint32_t dtype, float eps);

// gemv.hip
// how a GEMV launch reads its activations
enum : uint32_t {
    kXPlain = 0,    // row m of x
    kXGather = 1,   // row token(m) of x, the token id from the routing metadata (expert_assign fused)
    kXSiluMul = 2,  // x is [m, 2K]: silu(x[:, :K]) * x[:, K:] with expert_silu_mul's rounding
    kXDivide = 3,   // row m / x_div of x: the hybrid engine's project_id, whose routes share a token's row
};

// what route_token (route_device.hpp) takes: one token's routing by one wave
struct RouteTokenArgs {
    const void* logits;
    uint32_t logits_dtype;
    const float* bias;
    float* metadata;
    uint32_t experts, top_k, sigmoid, normalize;
    float eps, scaling;
    uint32_t rank_order;
    const void* gate_x;
    uint32_t gate_x_dtype;
    const float* gate_w;
    uint32_t hidden;
    float* shared_gate;
    float* ids_out;
    float* weights_out;
};

struct GemvArgs {
    uint32_t ggml_type;
    const void* w;        // packed [n, k] (per expert when metadata is set)
    const void* x;        // [m, k]
    void* y;              // [m, n]
    uint32_t n, k, m;
    uint32_t x_dtype, y_dtype;
    // expert form: when metadata != nullptr, row m of x uses expert
    // bits(metadata[3*m]) and weight rows [expert*n, expert*n + n)
    const float* metadata;
    uint32_t experts;
    int ksplit;           // 0 = automatic, else at least this many K segments
    uint32_t x_mode;      // kXPlain, kXGather or kXSiluMul
    uint32_t x_rows;      // rows of x (kXGather clamps the token id to it)
    uint32_t meta_stride; // floats per entry of `metadata`: 0 or 3 = {id, token, weight}, 1 = ids only
    uint32_t x_div;       // kXDivide: batch entries per row of x (0 = 1)
    // A shared expert riding in the same launch: the last shared_rows of the m batch entries
    // are tokens 0 .. shared_rows - 1 on the dense matrix shared_w [n, k], writing shared_y
    // [shared_rows, n]; they read row t of shared_x when set, else row t of x.  Null = none.
    const void* shared_w;
    uint32_t shared_rows;
    const void* shared_x;
    void* shared_y;
    // the streamed matrix-core kernel may take the launch (dense Q4_K or Q6_K, plain rows, rows that fit LDS)
    int stream;           // 0 never, 1 where it is the faster kernel, 2 wherever it can run
    int ring;             // fh_tuning::gemv_ring
    bool stream_own;      // the streamed Q4_K kernel's waves load their own super-blocks where tiles are <= 14 rows
    int cu_count;
    float* partials;      // scratch for K segments (gemv_plan says how much)
    uint32_t* counters;   // zeroed scratch, one word per (row tile, m)
    // One token whose routing has not run yet: every workgroup routes it first (one wave, the
    // bits of moe_route), takes its entry's expert from that, and workgroup 0 writes the records
    // to route->metadata for the launches that follow.  `metadata` is then only a non-null marker.
    const RouteTokenArgs* route;
};
struct GemvPlan {
    int bs, it;           // block slots per wave step, steps
    uint32_t segments, seg_len, rows_per_wg, tiles;
};
GemvPlan gemv_plan(uint32_t n, uint32_t k, uint32_t m, int forced_segments);
struct GemvScratch;
// planned: gemv_scratch(a)
const char* launch_gemv(hipStream_t s, const GemvArgs& a, const GemvScratch& planned);
// whether a launch with GemvArgs::route set exists for these rows and this router
bool gemv_routes(uint32_t n, uint32_t k, uint32_t experts, uint32_t top_k);

// gemv.hip: the down projection of a token's routed entries (and its shared expert) with
// expert_combine's weighted sum in the same launch; the bits of the two separate launches
struct ExpertDownCombineArgs {
    uint32_t ggml_type;
    const void* w;          // routed experts [experts][n, k]
    const void* w_shared;   // [n, k] or null
    const void* x;          // [tokens * top_k][2k] packed gate|up rows
    const void* x_shared;   // [tokens][2k]
    const float* metadata;  // [tokens * top_k][3]
    const float* shared_gate;
    void* y;                // [tokens][n]
    uint32_t n, k, tokens, top_k, experts, dtype;
};
bool expert_down_combine_fits(uint32_t ggml_type, uint32_t n, uint32_t k, uint32_t top_k, bool shared);
const char* launch_expert_down_combine(hipStream_t s, const ExpertDownCombineArgs& a);

// gemv_stream.hip: the Q4_K and Q6_K GEMV with LDS-direct weight loads and matrix-core dot products
struct StreamPlan {
    bool ok;              // the row length fits the kernel (LDS and per-wave block budget)
    uint32_t tile_rows;   // weight rows per workgroup (1..16)
    uint32_t tiles;
    uint32_t waves;       // waves per workgroup
    uint32_t row_stride;  // bytes between a tile's rows in LDS
    uint32_t lds_bytes;
    // rows too long for one tile are cut into K segments (grid.y), met through the scratch
    // partials and counters exactly as the FMA kernel's segments are
    uint32_t segments, seg_blocks;
    // the ring: a workgroup per compute unit, `tiles` of them per segment, with this many tiles in LDS (0: one tile per workgroup)
    uint32_t depth;
};
// any_size: also matrices so small that the FMA kernel is the faster one
StreamPlan gemv_stream_plan(uint32_t ggml_type, uint32_t n, uint32_t k, uint32_t m, int cu_count, bool any_size,
                            int forced_segments, int ring, bool f32_rows);
const char* launch_gemv_stream(hipStream_t s, const GemvArgs& a, const StreamPlan& plan);
// whether launch_gemv hands this launch to the streamed kernel, and its plan
bool gemv_takes_stream(const GemvArgs& a, StreamPlan* plan);
// K segments and row tiles of the kernel launch_gemv will run: what sizes the scratch.  The plan is made once per call (the
// smallest calls are bound by the host; here, for the scratch and for the launch it was made three times).
struct GemvScratch {
    uint32_t segments, tiles;
    StreamPlan stream;    // ok: the streamed kernel, with this plan
};
GemvScratch gemv_scratch(const GemvArgs& a);

// gemm_rows.hip: a few rows, f16 / bf16 on weights rounded to their type or f32 on exact f32 weights.  A workgroup's rows
// are a buffer of less than this (rows of more than sixty million elements go to the other kernels).
constexpr uint32_t kRowsBatchBytes = 0xf0000000u;
struct RowsPlan {
    uint32_t rows;            // rows a workgroup multiplies: 16 or 32
    uint32_t run_rows;        // rows of one launch; a larger batch is several, one after the other
    uint32_t groups;          // groups of `rows` rows of such a launch
    uint32_t k_waves;         // waves that share a tile's super-blocks
    uint32_t tiles;           // weight tiles of 16 rows per wave
    uint32_t tile_groups, segments, seg_blocks;
    size_t counters;          // scratch counter words of a launch (0: K is not cut)
    size_t partial_bytes;     // scratch for its partial sums (and operands)
    double estimate_us;
    bool pairs;               // f32 rows as pairs of f16 operands: gemm_pairs.hip
    size_t operand_bytes;     // ... which come first in the scratch
};
inline bool rows_batch_fits(const RowsPlan& plan, uint32_t k, uint32_t x_dtype) {
    return (uint64_t)plan.rows * k * dtype_bytes(x_dtype) <= kRowsBatchBytes;
}
RowsPlan gemm_rows_plan(uint32_t ggml_type, uint32_t n, uint32_t k, uint32_t m, uint32_t x_dtype, int cu_count);
// whether that plan's kernel, and not the FMA GEMV once per row, takes m exact f32 rows
bool f32_rows_pay(const RowsPlan& plan, uint32_t ggml_type, uint32_t n, uint32_t k, uint32_t m, int cu_count);

// gemm.hip
struct WidePlan {
    int nt;
    uint32_t cols, tiles_m, tiles_n;
    int rt;   // 32x32x16 form: row tiles of 32 per multiplying wave (2: 256-row tile, 1: 128-row tile)
    uint32_t segments, seg_blocks;   // 32x32x16 form: K segments
};
// Which of the tile forms would take a product of at least wide_min_rows rows, and the estimates.
struct TileChoice {
    bool made;
    bool wide_pays;      // the 16x16x32 form's workgroups cover at least half the chip
    WidePlan p32;        // the 32x32x16 form's tile, nt = 0 when it does not compete
    double us32, us16;
};

// How a product multiplies weights that were decoded first: its columns in one or two runs of tiles, a panel of each run at a time.
struct DecodedPlan {
    struct Run {
        uint32_t columns, tile, panel;   // of the matrix; of a tile; decoded at a time, a multiple of `tile`
    } run[2];
    int runs;              // 0: the weights are not decoded first
    uint32_t segments;     // K segments: 1, or 2 (one run then)
    size_t panel_bytes, sum_bytes;   // scratch: the largest panel, then the sums of one segment's tiles
};

struct GemmArgs {
    uint32_t ggml_type;
    const void* w;
    const void* x;        // [m, k] f16 or bf16
    void* y;              // [m, n]
    uint32_t n, k, m;
    uint32_t x_dtype, y_dtype;
    int cu_count;
    int wide_min_rows;   // smallest M that takes the 256-row tile
    int wide_shape;      // matrix instruction of the 256-row tile: 0 = 16x16x32, 1 = 32x32x16 where it wins, 2 = always
    int wide32_tile;     // 0 = chosen by shape; else 10 x (row tiles per wave) + column tiles of the 32x32x16 form
    int wide32_segments; // K segments of that form: 0 = by shape
    bool cut_tiles;      // its partial sums have room in the scratch (`partials`)
    TileChoice tile;     // made when first asked for; to be made again when cut_tiles changes
    int decoded_min_rows;      // rows from which the weights may be decoded once, in panels (0 = never)
    int decoded_tile;          // columns of the product's tile: 0 = by shape
    int decoded_segments;      // K segments of the product: 0 = by shape, else 1 or 2
    DecodedPlan decoded;       // set by gemm_takes_decoded; its panel and sums lie in `partials`
    int skinny_max_rows; // largest M that takes the register-dequant kernel where the rows-resident one is switched off
    // routed-expert form of the register-dequant kernel: w is [experts, n, k],
    // x and y rows are assignments, m is their count; tokens of expert e are
    // expert_order[expert_offsets[e] .. expert_offsets[e + 1])
    uint32_t experts;
    const uint32_t* expert_offsets;
    const uint32_t* expert_order;
    // routed form with the expert's rows resident in LDS (expert_rows_fit_lds): when set,
    // x is [x_rows, k] token rows and assignment a reads the row of its token,
    // gather_metadata[3a + 1], as expert_assign would have copied it
    const float* gather_metadata;
    uint32_t x_rows;
    // that kernel can carry a shared expert: tokens 0 .. shared_rows - 1 on the dense matrix
    // shared_w [n, k], reading row t of shared_x (null: row t of x, which then holds token
    // rows) and writing row t of shared_y
    const void* shared_w;
    uint32_t shared_rows;
    const void* shared_x;
    void* shared_y;
    bool x_rounds;   // routed form, rows resident, x_dtype f16: x and shared_x are f32 rows that the kernel rounds to f16
    // dense product: the rows are short enough to stay in LDS for the whole K (launch_gemm
    // then weighs launch_gemm_resident against the other kernels)
    bool rows_resident;
    bool use_resident;    // set by launch_gemm_resident only
    bool resident_switch; // rows_resident before the rows' length is looked at
    bool few_rows;        // the few-rows kernel may take the product (gemm_takes_rows)
    bool few_rows_always; // ... and does, whatever the estimates say
    RowsPlan rows_plan;   // set by gemm_takes_rows; its K segments and the tiles' meet in these:
    RowsPlan rows_else;   // where rows_plan is of pairs and has no room: the f32 instruction's, or none
    float* partials;
    uint32_t* counters;
    bool weight_ring;     // routed form, rows resident: Q4_K and Q6_K weights through LDS rings where they fit beside the rows
};
const char* launch_gemm(hipStream_t s, GemmArgs& a);
// whether launch_gemm hands this product to the few-rows kernel: fills a.rows_plan, whose partial sums and
// counters the caller then provides
bool gemm_takes_rows(GemmArgs& a);

// whether the weights are decoded into the scratch first (gemm_decoded.hip): fills a.decoded
bool gemm_takes_decoded(GemmArgs& a);
void launch_gemm_decoded(hipStream_t s, const GemmArgs& a);
double gemm_fused_estimate(GemmArgs& a);   // us of the kernel that decodes as it multiplies; 1e300: none is estimated
// scratch for the partial sums (or the panel) of the kernel launch_gemm would run (0: its K is not cut)
size_t gemm_partial_bytes(GemmArgs& a);

void launch_gemm_rows(hipStream_t s, const GemmArgs& a);   // gemm_rows.hip, by a.rows_plan

// gemm_pairs.hip: a batch of f32 rows on the f16 matrix instruction, exact integers times pairs of f16 values
// (whether it, and not the few-rows kernel, takes m of them)
bool pairs_pay(uint32_t ggml_type, uint32_t n, uint32_t k, uint32_t m);
RowsPlan gemm_pairs_plan(uint32_t n, uint32_t k, uint32_t m, int cu_count);
void launch_gemm_pairs(hipStream_t s, const GemmArgs& a);

// gemm_skinny.hip
const char* launch_gemm_skinny(hipStream_t s, const GemmArgs& a);
// dense [m, k] x [n, k]^T with 16 or 32 rows at a time resident in LDS; needs expert_rows_fit_lds(k, 1, 1)
const char* launch_gemm_resident(hipStream_t s, const GemmArgs& a);
// whether the routed form keeps an expert's activation rows of width k in LDS,
// which is the kernel that takes the gathered input form
bool expert_rows_fit_lds(uint32_t k, uint32_t m, uint32_t experts);

// moe.hip
// what the hybrid engine's router adds: selection order kept, shared-expert gate
struct RouteExtras {
    uint32_t rank_order = 0;
    const void* gate_x = nullptr;      // [tokens, hidden] activations the gate vector is dotted with
    uint32_t gate_x_dtype = 0;
    const float* gate_w = nullptr;     // [hidden], or null: the gate is 1
    uint32_t hidden = 0;
    float* shared_gate = nullptr;      // [tokens], or null: no gate output
    float* ids_out = nullptr;          // [tokens, top_k] expert ids as u32 bits, or null
    float* weights_out = nullptr;      // [tokens, top_k] route weights, or null
};
const char* launch_moe_route(hipStream_t s, const void* logits, uint32_t logits_dtype,
                             const float* bias, float* metadata, uint32_t tokens,
                             const fh_routing_policy& policy, const RouteExtras& extras);
// the hybrid engine's stages over plain id / weight arrays (h_moe_map, h_moe_gather, h_moe_combine)
const char* launch_moe_map(hipStream_t s, const uint32_t* ids, uint32_t experts, uint32_t routes, uint32_t* offsets,
                           uint32_t* sorted, uint32_t* position);
const char* launch_moe_gather_sorted(hipStream_t s, const void* x, const uint32_t* sorted, void* out, uint32_t routes,
                                     uint32_t used, uint32_t tokens, uint32_t row_bytes);
const char* launch_hybrid_combine(hipStream_t s, const float* down, const float* weights, const uint32_t* position,
                                  const float* shared, const float* shared_gate, float* out, uint32_t hidden,
                                  uint32_t used, uint32_t tokens, uint32_t rows);
const char* launch_expert_group(hipStream_t s, const float* metadata, uint32_t assignments,
                                uint32_t experts, uint32_t* offsets, uint32_t* order, void* y,
                                uint32_t row_bytes);
const char* launch_expert_assign(hipStream_t s, const void* hidden, const float* metadata,
                                 void* out, uint32_t assignments, uint32_t row_bytes, uint32_t tokens);
const char* launch_expert_silu_mul(hipStream_t s, const void* in, void* out, uint32_t assignments,
                                   uint32_t intermediate, uint32_t in_dtype, uint32_t out_dtype);
void launch_expert_silu_mul_pair(hipStream_t s, const void* in, const void* in2, void* out, uint32_t rows,
                                 uint32_t rows2, uint32_t intermediate, uint32_t dtype);
const char* launch_expert_combine(hipStream_t s, const void* in, const float* metadata, void* out,
                                  uint32_t tokens, uint32_t hidden, uint32_t top_k,
                                  uint32_t in_dtype, uint32_t out_dtype, const void* shared,
                                  const float* shared_gate);

}  // namespace fh
