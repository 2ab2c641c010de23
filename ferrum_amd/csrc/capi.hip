// C ABI of the gfx950 backend (see include/ferrum_hip.h): objects, validation
// and kernel selection.  Argument checks mirror the reference's operator
// methods (src/ops/transformer.rs:96-297, src/ops/mod.rs:23-609) and its
// binding checks (src/metal/mod.rs:840-897): shapes, ownership, bounds,
// alignment and input/output aliasing are rejected before anything launches.
#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <mutex>
#include <cstring>
#include <new>
#include <vector>

#include "internal.hpp"

namespace fh {

static thread_local std::string g_last_error;

fh_status fail(fh_status code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_last_error = buf;
    return code;
}

fh_status hip_fail(hipError_t err, const char* what) {
    fh_status code = err == hipErrorOutOfMemory ? FH_ERR_ALLOCATION : FH_ERR_DISPATCH;
    return fail(code, "%s: %s", what, hipGetErrorString(err));
}

namespace {

#define FH_HIP(expr)                                        \
    do {                                                    \
        hipError_t _e = (expr);                             \
        if (_e != hipSuccess) return hip_fail(_e, #expr);   \
    } while (0)

struct Range {
    const uint8_t* begin;
    size_t bytes;
};

bool overlaps(const Range& a, const Range& b) {
    return a.begin < b.begin + b.bytes && b.begin < a.begin + a.bytes;
}

// Resolves a view to a device pointer after ownership, bounds and alignment
// checks.  `elements` is the number of dtype-sized elements the op touches.
fh_status resolve(const fh_device* device, const fh_view* view, uint64_t elements, const char* what,
                  Range* out, size_t alignment = 16) {
    if (view == nullptr || view->buffer == nullptr)
        return fail(FH_ERR_RANGE, "%s: null view", what);
    if (view->dtype > FH_BF16) return fail(FH_ERR_DTYPE, "%s: unknown dtype %u", what, view->dtype);
    if (view->buffer->device != device) {
        g_last_error = std::string(what) + ": buffer belongs to another device";
        return FH_ERR_DEVICE_MISMATCH;
    }
    uint64_t bytes = elements * dtype_bytes(view->dtype);
    if (view->offset > view->buffer->bytes || bytes > view->buffer->bytes - view->offset)
        return fail(FH_ERR_RANGE, "%s: view [%zu, +%llu) exceeds buffer of %zu bytes", what,
                    view->offset, (unsigned long long)bytes, view->buffer->bytes);
    if (view->offset % alignment != 0)
        return fail(FH_ERR_RANGE, "%s: offset %zu is not %zu-byte aligned", what, view->offset,
                    alignment);
    out->begin = static_cast<const uint8_t*>(view->buffer->ptr) + view->offset;
    out->bytes = (size_t)bytes;
    return FH_OK;
}

bool fits_u32(uint64_t v) { return v <= 0xffffffffull; }

// A block back to the system; hipFree waits for all work on the block's GPU when it succeeds.
bool give_back(const fh_device* d, void* block) {
    int current = d->ordinal;
    (void)hipGetDevice(&current);
    if (current != d->ordinal) (void)hipSetDevice(d->ordinal);
    const hipError_t e = hipFree(block);
    if (e != hipSuccess) (void)hipGetLastError();
    if (current != d->ordinal) (void)hipSetDevice(current);
    return e == hipSuccess;
}

// Gives back what the device keeps for buffers to come; whether that was anything.  A device that is
// recording keeps its blocks: neither a wait on its stream nor a free may fall into a recording.
bool drain(fh_device* d) {
    return d->freed.drain([d] { return !d->capturing; }, [d] { (void)hipStreamSynchronize(d->stream); },
                          [d](void* block) { return give_back(d, block); });
}

// Every device object between fh_device_create and fh_device_destroy.
std::mutex g_live_lock;
fh_device* g_live = nullptr;

void enter_live(fh_device* d) {
    std::lock_guard<std::mutex> hold(g_live_lock);
    d->next_live = g_live;
    g_live = d;
}

void leave_live(fh_device* d) {
    std::lock_guard<std::mutex> hold(g_live_lock);
    for (fh_device** at = &g_live; *at != nullptr; at = &(*at)->next_live)
        if (*at == d) {
            *at = d->next_live;
            return;
        }
}

// Gives back what the device objects on this GPU keep for themselves; whether that was anything.
bool drain_pools(int ordinal) {
    bool any = false;
    std::lock_guard<std::mutex> hold(g_live_lock);
    for (fh_device* d = g_live; d != nullptr; d = d->next_live) {
        if (d->ordinal != ordinal) continue;
        any = drain(d) || any;
    }
    return any;
}

// A block from the system; above the device's allocation_limit_bytes the request is one that no GPU has room for.
hipError_t request(const fh_device* d, void** out, size_t bytes) {
    const uint64_t limit = (uint64_t)d->tuning.allocation_limit_bytes;
    return hipMalloc(out, limit != 0 && bytes > limit ? (size_t)1 << 60 : bytes);
}

// Memory from the system; what the pools on this GPU hold is given back when there is none.
hipError_t allocate(fh_device* d, void** out, size_t bytes) {
    hipError_t e = request(d, out, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        if (drain_pools(d->ordinal)) e = request(d, out, bytes);
        if (e == hipErrorOutOfMemory) (void)hipGetLastError();   // the caller's to report: a launch may follow instead
    }
    return e;
}

constexpr size_t kScratchCounterBytes = fh_device::kCounterWords * sizeof(uint32_t);

bool scratch_holds(const fh_device* d, size_t data_bytes) {
    return d->scratch != nullptr && d->scratch_bytes >= kScratchCounterBytes + data_bytes;
}

// A new block for a scratch that holds less; the old one stays until the new one is there.  Recorded executions carry the
// scratch address in their kernel arguments, so a block that is outgrown while any of them is alive is kept (they replay on
// it unchanged) and freed with the last one.
fh_status grow_scratch(fh_device* d, size_t data_bytes, bool optional) {
    const size_t asked = std::max(data_bytes, fh_device::kScratchFloor);
    // twice the old data area, so that the blocks kept for recordings add up to less than the live one and growth in small
    // steps ends; but no more than the largest of the areas that only save time unless a request itself is larger
    const size_t old_data = d->scratch != nullptr ? d->scratch_bytes - kScratchCounterBytes : 0;
    size_t data = asked <= fh_device::kScratchOptional ? std::max(asked, std::min(2 * old_data, fh_device::kScratchOptional))
                  : d->live_graphs > 0                 ? std::max(asked, 2 * old_data)
                                                       : asked;
    void* block = nullptr;
    hipError_t e = allocate(d, &block, kScratchCounterBytes + data);
    if (e == hipErrorOutOfMemory && data > asked) {
        data = asked;
        e = allocate(d, &block, kScratchCounterBytes + data);
    }
    if (e == hipErrorOutOfMemory && !optional && d->scratch != nullptr && d->live_graphs == 0) {
        // the old block may be what is missing; if that is not it either, the device gets its smallest one back
        FH_HIP(hipStreamSynchronize(d->stream));
        (void)hipFree(d->scratch);
        d->scratch = nullptr;
        d->scratch_bytes = 0;
        e = allocate(d, &block, kScratchCounterBytes + data);
        if (e == hipErrorOutOfMemory && data > fh_device::kScratchFloor) {
            const fh_status st = grow_scratch(d, 0, false);
            if (st != FH_OK) return st;
        }
    }
    if (e != hipSuccess)
        return fail(FH_ERR_ALLOCATION, "hipMalloc(%zu): %s", kScratchCounterBytes + data, hipGetErrorString(e));
    e = hipMemsetAsync(block, 0, kScratchCounterBytes, d->stream);
    if (e == hipSuccess && d->scratch != nullptr && d->live_graphs == 0) e = hipStreamSynchronize(d->stream);
    if (e != hipSuccess) {
        (void)hipFree(block);
        return hip_fail(e, "scratch");
    }
    if (d->scratch != nullptr) {
        if (d->live_graphs > 0) d->retired_scratch.push_back(d->scratch);
        else (void)hipFree(d->scratch);
    }
    d->scratch = block;
    d->scratch_bytes = kScratchCounterBytes + data;
    return FH_OK;
}

// Device scratch: kCounterWords zeroed counter words followed by a data area of at least `data_bytes`.
fh_status ensure_scratch(fh_device* d, size_t data_bytes) {
    if (scratch_holds(d, data_bytes)) return FH_OK;
    if (d->capturing)
        return fail(FH_ERR_SYNCHRONIZATION, "device scratch must grow: run the operator once before recording it");
    return grow_scratch(d, data_bytes, false);
}

// Whether the scratch can be brought to `data_bytes` now: it does not grow while an execution is being
// recorded.  Kernels that only save time by using it leave such a call to those that need none.
bool scratch_available(const fh_device* d, size_t data_bytes) { return !d->capturing || scratch_holds(d, data_bytes); }

// The same for such a kernel's own needs: FH_ERR_ALLOCATION where there is no room.  A GPU that had none is asked again
// only after some calls: each request that fails empties the pools, which waits for the stream.
fh_status optional_scratch(fh_device* d, size_t data_bytes) {
    constexpr uint32_t kCallsBetween = 256;
    if (scratch_holds(d, data_bytes)) return FH_OK;
    if (d->capturing) return FH_ERR_ALLOCATION;
    if (d->scratch_refused != 0 && data_bytes >= d->scratch_refused && d->scratch_wait > 0) {
        --d->scratch_wait;
        return FH_ERR_ALLOCATION;
    }
    const fh_status st = grow_scratch(d, data_bytes, true);
    if (st == FH_ERR_ALLOCATION) {
        d->scratch_refused = data_bytes;
        d->scratch_wait = kCallsBetween;
    } else if (data_bytes >= d->scratch_refused) {
        d->scratch_refused = 0;
    }
    return st;
}

// Brings the scratch back to its smallest size, unless recorded executions carry its address.
fh_status shrink_scratch(fh_device* d) {
    if (d->capturing) return fail(FH_ERR_SYNCHRONIZATION, "not available while an execution is being recorded");
    if (d->live_graphs > 0 || d->scratch_bytes <= kScratchCounterBytes + fh_device::kScratchFloor) return FH_OK;
    FH_HIP(hipStreamSynchronize(d->stream));
    (void)hipFree(d->scratch);
    d->scratch = nullptr;
    d->scratch_bytes = 0;
    return grow_scratch(d, 0, false);
}

// A block the library owns for its own temporaries (it holds no count on the device), grown like
// the scratch: outside recordings only, by at least 2x, old blocks kept for the recorded executions
// that carry their address.
fh_status ensure_block(fh_device* d, fh_buffer*& slot, size_t bytes, const char* what) {
    if (slot != nullptr && slot->bytes >= bytes) return FH_OK;
    if (d->capturing)
        return fail(FH_ERR_SYNCHRONIZATION, "%s must grow: run the call once before recording it", what);
    FH_HIP(hipStreamSynchronize(d->stream));
    if (slot == nullptr) {
        slot = new (std::nothrow) fh_buffer();
        if (slot == nullptr) return fail(FH_ERR_ALLOCATION, "out of host memory");
        slot->device = d;
    }
    if (bytes < 2 * slot->bytes) bytes = 2 * slot->bytes;
    if (slot->ptr) {
        if (d->live_graphs > 0) d->retired_scratch.push_back(slot->ptr);
        else (void)hipFree(slot->ptr);
    }
    slot->ptr = nullptr;
    slot->bytes = 0;
    hipError_t e = allocate(d, &slot->ptr, bytes);
    if (e != hipSuccess) return fail(FH_ERR_ALLOCATION, "hipMalloc(%zu): %s", bytes, hipGetErrorString(e));
    slot->bytes = bytes;
    return FH_OK;
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// ---- matrices whose rows are stored padded (Q8_0 rows of 32 n weights, n not a multiple of 8) ----
// An entry point that meets one runs on the matrix as it is stored (rows of stored_cols weights,
// the added blocks empty) and on its activations rewritten to that width, zeros in the added
// columns, in a block of the device's own.  Everything behind that point is the ordinary path.
fh_qmatrix as_stored(const fh_qmatrix* w) {
    fh_qmatrix m = *w;
    m.cols = w->stored_cols;
    return m;
}

struct PaddedActivations {
    struct Item {
        const fh_view* x;
        uint64_t pieces;   // rows x parts: runs of `cols` elements
        const char* what;
        fh_view* out;
        Range range;
    };
    fh_device* device;
    uint64_t cols, stored;
    Item items[2];
    int count = 0;
    PaddedActivations(fh_device* d, const fh_qmatrix* w) : device(d), cols(w->cols), stored(w->stored_cols) {}
    void add(const fh_view* x, uint64_t pieces, const char* what, fh_view* out) {
        items[count++] = Item{x, pieces, what, out, Range{nullptr, 0}};
    }
    // checks the views, then writes the padded copies and points `out` at them
    fh_status run() {
        size_t at = 0, offsets[2] = {0, 0};
        for (int i = 0; i < count; ++i) {
            Item& it = items[i];
            if (!fits_u32(it.pieces * stored)) return fail(FH_ERR_SHAPE, "index does not fit in 32 bits");
            fh_status st = resolve(device, it.x, it.pieces * cols, it.what, &it.range);
            if (st != FH_OK) return st;
            offsets[i] = at;
            at += align256((size_t)(it.pieces * stored) * dtype_bytes(it.x->dtype));
        }
        fh_status st = ensure_block(device, device->padded_rows, at, "the block for padded activations");
        if (st != FH_OK) return st;
        for (int i = 0; i < count; ++i) {
            const Item& it = items[i];
            launch_pad_rows(device->stream, it.range.begin, static_cast<uint8_t*>(device->padded_rows->ptr) + offsets[i],
                            (size_t)it.pieces, (size_t)cols, (size_t)stored, dtype_bytes(it.x->dtype));
            *it.out = fh_view{device->padded_rows, offsets[i], it.x->dtype};
        }
        FH_HIP(hipGetLastError());
        return FH_OK;
    }
    // an output may not alias the activations as the caller passed them
    fh_status keep_apart(const fh_view* y, uint64_t elements, const char* what, const char* message) const {
        Range yr;
        fh_status st = resolve(device, y, elements, what, &yr);
        if (st != FH_OK) return st;
        for (int i = 0; i < count; ++i)
            if (overlaps(items[i].range, yr)) return fail(FH_ERR_RANGE, "%s", message);
        return FH_OK;
    }
};

uint32_t* scratch_counters(fh_device* d) { return static_cast<uint32_t*>(d->scratch); }
uint8_t* scratch_data(fh_device* d) {
    return static_cast<uint8_t*>(d->scratch) + fh_device::kCounterWords * sizeof(uint32_t);
}

// Points a GEMV launch that cuts K into segments at the device scratch
// (partial sums and one zeroed counter word per row tile and batch row).  `plan` is gemv_scratch(a) and stays so.
fh_status prepare_gemv(fh_device* d, GemvArgs& a, GemvScratch& plan) {
    if (a.ring != 0 && plan.segments > 1 && !scratch_available(d, (size_t)plan.segments * a.m * a.n * sizeof(float))) {
        a.ring = 0;   // the ring may want more segments than the scratch of a recording has room for
        plan = gemv_scratch(a);
    }
    if (plan.segments > 1) {
        if ((uint64_t)plan.tiles * a.m > fh_device::kCounterWords)
            return fail(FH_ERR_SHAPE, "projection needs %llu row tiles, more than the K-split scratch holds",
                        (unsigned long long)plan.tiles * a.m);
        fh_status st = ensure_scratch(d, (size_t)plan.segments * a.m * a.n * sizeof(float));
        if (st != FH_OK) return st;
        a.partials = reinterpret_cast<float*>(scratch_data(d));
        a.counters = scratch_counters(d);
    }
    return FH_OK;
}

// Runs a GEMV launch of any batch size: the batch is cut into runs that fit the grid's z
// extent and, where K is cut into segments, the counter words (one per row tile and batch
// entry).  A launch that carries a shared expert is not cut.
fh_status run_gemv(fh_device* d, GemvArgs a, const char** name) {
    GemvScratch plan = gemv_scratch(a);
    uint64_t most = 65535u;
    if (plan.segments > 1 && plan.tiles > 0) most = std::min<uint64_t>(most, fh_device::kCounterWords / plan.tiles);
    if (a.x_mode == kXDivide && a.x_div > 1) most -= most % a.x_div;   // the routes of a token stay together
    if (a.m <= most || a.shared_w != nullptr || most == 0) {
        fh_status st = prepare_gemv(d, a, plan);
        if (st != FH_OK) return st;
        if (a.m > 65535u) return fail(FH_ERR_SHAPE, "batch of %u entries exceeds the launch grid", a.m);
        *name = launch_gemv(d->stream, a, plan);
        return FH_OK;
    }
    const uint32_t total = a.m;
    const size_t x_row = (size_t)a.k * dtype_bytes(a.x_dtype) * (a.x_mode == kXSiluMul ? 2 : 1);
    const size_t y_row = (size_t)a.n * dtype_bytes(a.y_dtype);
    const uint32_t stride = a.meta_stride == 0 ? 3u : a.meta_stride;
    for (uint32_t first = 0; first < total; first += (uint32_t)most) {
        GemvArgs part = a;
        part.m = std::min<uint32_t>((uint32_t)most, total - first);
        part.y = static_cast<uint8_t*>(a.y) + first * y_row;
        if (a.metadata != nullptr) part.metadata = a.metadata + (size_t)first * stride;
        if (a.x_mode == kXPlain || a.x_mode == kXSiluMul) {
            part.x = static_cast<const uint8_t*>(a.x) + first * x_row;
            part.x_rows = part.m;
        } else if (a.x_mode == kXDivide) {
            const uint32_t div = a.x_div == 0 ? 1u : a.x_div;
            part.x = static_cast<const uint8_t*>(a.x) + (size_t)(first / div) * x_row;
            part.x_rows = part.m / div;
        }   // kXGather reads the token row named by each entry's metadata: x stays whole
        GemvScratch part_plan = gemv_scratch(part);
        fh_status st = prepare_gemv(d, part, part_plan);
        if (st != FH_OK) return st;
        *name = launch_gemv(d->stream, part, part_plan);
    }
    return FH_OK;
}

// Frees device memory now, or after the recording in progress has ended.
void release_memory(fh_device* d, void* ptr) {
    if (ptr == nullptr) return;
    if (d != nullptr && d->closed) {
        (void)hipFree(ptr);   // synchronizes by itself; the stream no longer exists
        return;
    }
    if (d != nullptr && d->capturing) {
        d->deferred_frees.push_back(ptr);
        return;
    }
    if (d != nullptr) (void)hipStreamSynchronize(d->stream);
    (void)hipFree(ptr);
}

// One object created on the device is gone (or the caller's handle is); the last one frees it.
void drop_device_handle(fh_device* d) {
    if (d != nullptr && --d->handles == 0) delete d;
}

void drain_deferred(fh_device* d) {
    if (d->deferred_frees.empty() && d->deferred_graphs.empty()) return;
    (void)hipStreamSynchronize(d->stream);
    for (void* ptr : d->deferred_frees) (void)hipFree(ptr);
    for (auto& g : d->deferred_graphs) {
        (void)hipGraphExecDestroy(g.first);
        (void)hipGraphDestroy(g.second);
    }
    d->deferred_frees.clear();
    d->deferred_graphs.clear();
}

constexpr struct {
    const char* name;
    int64_t fh_tuning::*value;
} kTuningKeys[] = {
    {"k_quant_gemv_ksplit", &fh_tuning::k_quant_gemv_ksplit},
    {"gemm_min_rows", &fh_tuning::gemm_min_rows},
    {"gemm_wide_shape", &fh_tuning::gemm_wide_shape},
    {"gemm_wide32_tile", &fh_tuning::gemm_wide32_tile},
    {"gemm_wide32_segments", &fh_tuning::gemm_wide32_segments},
    {"gemm_decoded_min_rows", &fh_tuning::gemm_decoded_min_rows},
    {"gemm_decoded_tile", &fh_tuning::gemm_decoded_tile},
    {"gemm_decoded_segments", &fh_tuning::gemm_decoded_segments},
    {"gemm_wide_min_rows", &fh_tuning::gemm_wide_min_rows},
    {"gemm_skinny_max_rows", &fh_tuning::gemm_skinny_max_rows},
    {"expert_grouped_min_assignments", &fh_tuning::expert_grouped_min_assignments},
    {"moe_fold_route", &fh_tuning::moe_fold_route},
    {"gemm_few_tiles_split", &fh_tuning::gemm_few_tiles_split},
    {"moe_fold_combine", &fh_tuning::moe_fold_combine},
    {"gemm_resident", &fh_tuning::gemm_resident},
    {"gemv_ring", &fh_tuning::gemv_ring},
    {"gemv_stream_own_loads", &fh_tuning::gemv_stream_own_loads},
    {"expert_weight_ring", &fh_tuning::expert_weight_ring},
    {"gemv_stream", &fh_tuning::gemv_stream},
    {"moe_routing_temporary_limit", &fh_tuning::moe_routing_temporary_limit},
    {"gemm_f32_min_rows", &fh_tuning::gemm_f32_min_rows},
    {"allocation_limit_bytes", &fh_tuning::allocation_limit_bytes},
    {"probe_read_form", &fh_tuning::probe_read_form},
};

// the switch of that name, or null
template <class Device>
auto tuning_of(Device* d, const char* key) -> decltype(&(d->tuning.gemm_min_rows)) {
    for (const auto& k : kTuningKeys)
        if (std::strcmp(k.name, key) == 0) return &(d->tuning.*k.value);
    return nullptr;
}

// ---- freed blocks kept for the next buffers ----------------------------------------------

// Blocks come in sizes a quarter of a power of two apart (4 KiB at least), so that a batch a little larger
// or smaller finds them.
size_t block_capacity(size_t bytes) {
    if (bytes > FreedBlocks::kPoolBlockBytes) return bytes;
    size_t step = 4096;
    while (step * 8 < bytes) step *= 2;
    return (bytes + step - 1) / step * step;
}

hipError_t take_block(fh_device* d, size_t capacity, void** out) {
    return d->freed.take(capacity, out) ? hipSuccess : allocate(d, out, capacity);
}

// Keeps a freed buffer's block; false: the caller frees it.  Nothing waits: whatever the
// library still has to do with the block comes before the next buffer's work on the stream.  A block whose
// address the caller has been given may be in use elsewhere and waits, with others, until it cannot be.
bool keep_block(fh_device* d, const fh_buffer& buffer) {
    const auto may = [d] { return !d->closed && !d->capturing; };
    if (buffer.capacity > FreedBlocks::kPoolBlockBytes) return false;
    if (buffer.exposed) {
        bool full = false;
        if (!d->freed.gather(buffer.capacity, buffer.ptr, may, &full)) return false;
        if (full) d->freed.settle(may, [d](void* block) { return give_back(d, block); });
        return true;
    }
    if (!d->freed.fits(buffer.capacity)) drain(d);   // it holds sizes that are no longer asked for
    return d->freed.keep(buffer.capacity, buffer.ptr, may);
}

}  // namespace
}  // namespace fh

using namespace fh;

// Scratch of the entry point that allocates nothing: the K-segment partial sums and the
// row-tile counters of the GEMV.  Every device the library runs on holds its own copy of
// the array at its own address for the life of the process; `scratch` itself is only the
// host-side name of the symbol, the device address comes from hipGetSymbolAddress.
constexpr size_t kFixedCounterWords = 4096;
constexpr size_t kFixedScratchBytes = 1u << 20;   // 16 KiB of counters, then partial sums
static __device__ __align__(256) unsigned char scratch[kFixedScratchBytes];

static_assert(kXDivide > FH_INPUT_SILU_MUL, "the row-divide mode is internal: it has no public input form");
static_assert(kXPlain == FH_INPUT_ROWS && kXGather == FH_INPUT_GATHER && kXSiluMul == FH_INPUT_SILU_MUL,
              "the kernel's input modes are the ABI's input forms");

extern "C" {

const char* fh_last_error(void) { return g_last_error.c_str(); }

fh_status fh_device_create(int32_t ordinal, fh_device** out) {
    if (out == nullptr) return fail(FH_ERR_PARAMETER, "fh_device_create: null output");
    *out = nullptr;
    int count = 0;
    FH_HIP(hipGetDeviceCount(&count));
    if (ordinal < 0 || ordinal >= count)
        return fail(FH_ERR_DISPATCH, "no HIP device %d (found %d)", ordinal, count);
    FH_HIP(hipSetDevice(ordinal));
    fh_device* d = new (std::nothrow) fh_device();
    if (d == nullptr) return fail(FH_ERR_ALLOCATION, "out of host memory");
    d->ordinal = ordinal;
    hipError_t e = hipGetDeviceProperties(&d->props, ordinal);
    if (e != hipSuccess) {
        delete d;
        return hip_fail(e, "hipGetDeviceProperties");
    }
    if (std::strncmp(d->props.gcnArchName, "gfx950", 6) != 0) {
        fh_status st = fail(FH_ERR_DISPATCH, "kernels are built for gfx950 only; device %d is %s",
                            ordinal, d->props.gcnArchName);
        delete d;
        return st;
    }
    e = hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        delete d;
        return hip_fail(e, "hipStreamCreateWithFlags");
    }
    fh_status st = ensure_scratch(d, 0);
    if (st == FH_OK) {
        // This device's address of the fixed scratch (the device is current).  Its counters are set to zero
        // once per GPU and process: launches leave them at zero, and a second handle on a GPU whose first
        // handle has a K-split launch in flight must not reset that launch's tickets.
        void* fixed = nullptr;
        e = hipGetSymbolAddress(&fixed, HIP_SYMBOL(scratch));
        if (e == hipSuccess) {
            static std::mutex zero_lock;
            static bool zeroed[256] = {};
            std::lock_guard<std::mutex> hold(zero_lock);
            if (ordinal < 256 && !zeroed[ordinal]) {
                e = hipMemsetAsync(fixed, 0, kFixedCounterWords * sizeof(uint32_t), d->stream);
                if (e == hipSuccess) e = hipStreamSynchronize(d->stream);
                if (e == hipSuccess) zeroed[ordinal] = true;
            }
        }
        if (e != hipSuccess) st = hip_fail(e, "fixed scratch");
        d->fixed_scratch = fixed;
    }
    if (st != FH_OK) {
        if (d->scratch) (void)hipFree(d->scratch);
        (void)hipStreamDestroy(d->stream);
        delete d;
        return st;
    }
    enter_live(d);
    *out = d;
    return FH_OK;
}

void fh_device_destroy(fh_device* device) {
    if (device == nullptr) return;
    (void)hipSetDevice(device->ordinal);
    if (device->closed) return;
    // what was put off during a recording goes first, while the stream it waits on exists
    if (device->capturing) {
        hipGraph_t abandoned = nullptr;
        (void)hipStreamEndCapture(device->stream, &abandoned);
        if (abandoned) (void)hipGraphDestroy(abandoned);
        device->capturing = false;
    }
    drain_deferred(device);
    leave_live(device);
    {
        std::lock_guard<std::mutex> alone(device->freed.settling);
        std::lock_guard<std::mutex> hold(device->freed.lock);
        device->closed = true;   // buffers freed from here on are not kept
    }
    drain(device);
    if (device->stream) {
        (void)hipStreamSynchronize(device->stream);
        (void)hipStreamDestroy(device->stream);
        device->stream = nullptr;
    }
    if (device->scratch) (void)hipFree(device->scratch);
    if (device->workspace) {
        if (device->workspace->ptr) (void)hipFree(device->workspace->ptr);
        delete device->workspace;
        device->workspace = nullptr;
    }
    if (device->padded_rows) {
        if (device->padded_rows->ptr) (void)hipFree(device->padded_rows->ptr);
        delete device->padded_rows;
        device->padded_rows = nullptr;
    }
    for (void* old : device->retired_scratch) (void)hipFree(old);
    device->retired_scratch.clear();
    device->scratch = nullptr;
    device->scratch_bytes = 0;
    drop_device_handle(device);
}

fh_status fh_device_properties(const fh_device* device, fh_device_props* out) {
    if (device == nullptr || out == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    std::memset(out, 0, sizeof(*out));
    std::snprintf(out->name, sizeof(out->name), "%s", device->props.name);
    if (out->name[0] == '\0')   // some driver stacks leave the marketing name empty
        std::snprintf(out->name, sizeof(out->name), "%.40s, %d CUs, %.0f GiB", device->props.gcnArchName,
                      device->props.multiProcessorCount, (double)device->props.totalGlobalMem / (1 << 30));
    std::snprintf(out->arch, sizeof(out->arch), "%s", device->props.gcnArchName);
    out->compute_units = device->props.multiProcessorCount;
    out->wavefront = device->props.warpSize;
    out->clock_khz = device->props.clockRate;
    out->memory_clock_khz = device->props.memoryClockRate;
    out->memory_bus_bits = device->props.memoryBusWidth;
    out->lds_bytes_per_block = (int32_t)device->props.sharedMemPerBlock;
    out->global_bytes = device->props.totalGlobalMem;
    out->l2_bytes = (uint64_t)device->props.l2CacheSize;
    return FH_OK;
}

fh_status fh_synchronize(fh_device* device) {
    if (device && device->capturing) return fail(FH_ERR_SYNCHRONIZATION, "not available while an execution is being recorded");
    if (device == nullptr) return fail(FH_ERR_PARAMETER, "null device");
    hipError_t e = hipStreamSynchronize(device->stream);
    if (e != hipSuccess) return fail(FH_ERR_SYNCHRONIZATION, "stream: %s", hipGetErrorString(e));
    return FH_OK;
}

const char* fh_last_operation(const fh_device* device) {
    return device ? device->last_operation : "";
}

void* fh_device_stream(fh_device* device) { return device ? device->stream : nullptr; }

fh_status fh_set_tuning(fh_device* device, const char* key, int64_t value) {
    if (device == nullptr || key == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (std::strcmp(key, "held_pool_bytes") == 0 && value == 0) {
        FH_HIP(hipSetDevice(device->ordinal));
        drain_pools(device->ordinal);
        return FH_OK;
    }
    if (std::strcmp(key, "held_scratch_bytes") == 0 && value == 0) {
        FH_HIP(hipSetDevice(device->ordinal));
        return shrink_scratch(device);
    }
    int64_t* const setting = tuning_of(device, key);
    if (setting == nullptr) return fail(FH_ERR_PARAMETER, "unknown tuning key %s", key);
    std::string k(key);
    bool ok = true;
    if (k == "k_quant_gemv_ksplit") {
        // set_k_quant_gemv_ksplit: 0 or a power of two up to 8
        ok = value == 0 || value == 1 || value == 2 || value == 4 || value == 8;
    } else if (k == "gemm_min_rows") {
        ok = value >= 2;
    } else if (k == "gemm_resident" || k == "moe_fold_combine" || k == "moe_fold_route") {
        ok = value == 0 || value == 1;
    } else if (k == "gemv_stream_own_loads" || k == "expert_weight_ring") {
        ok = value == 0 || value == 1;
    } else if (k == "gemv_stream" || k == "gemv_ring" || k == "gemm_few_tiles_split" ||
               k == "gemm_decoded_segments") {
        ok = value >= 0 && value <= 2;
    } else if (k == "gemm_wide_shape") {
        ok = value >= 0 && value <= 2;
    } else if (k == "gemm_wide32_tile") {
        ok = value == 0 || value == 12 || value == 13 || value == 14 || value == 15 || value == 24 || value == 25;
    } else if (k == "gemm_wide32_segments") {
        ok = value >= 0 && value <= 8;
    } else if (k == "gemm_decoded_min_rows") {
        ok = value >= 0 && value <= INT32_MAX;
    } else if (k == "gemm_decoded_tile") {
        ok = value == 0 || value == 192 || value == 256 || value == 320;
    } else if (k == "gemm_wide_min_rows") {
        ok = value >= 1;
    } else if (k == "gemm_skinny_max_rows") {
        ok = value >= 0 && value <= 64;
    } else if (k == "expert_grouped_min_assignments" || k == "allocation_limit_bytes") {
        ok = value >= 0;
    } else if (k == "gemm_f32_min_rows") {
        ok = value == 0 || value >= 2;
    } else if (k == "probe_read_form") {
        ok = value == 0 || value == 25604 || value == 25608 || value == 25616 || value == 51204 || value == 51208 ||
             value == 102404 || value == 102408 || value == 1025608 || value == 1025616 || value == 1051208;
    } else if (k == "moe_routing_temporary_limit") {
        // set_moe_routing_temporary_limit (src/metal/legacy.rs:523-531): positive, on an idle device
        ok = value > 0 && !device->capturing;
    }
    if (!ok) return fail(FH_ERR_PARAMETER, "value %lld is out of range for %s", (long long)value, key);
    *setting = value;
    return FH_OK;
}

fh_status fh_get_tuning(const fh_device* device, const char* key, int64_t* value) {
    if (device == nullptr || key == nullptr || value == nullptr)
        return fail(FH_ERR_PARAMETER, "null argument");
    if (std::strcmp(key, "held_scratch_bytes") == 0) {
        *value = (int64_t)device->scratch_bytes;
        return FH_OK;
    }
    if (std::strcmp(key, "retired_scratch_blocks") == 0) {
        *value = (int64_t)device->retired_scratch.size();
        return FH_OK;
    }
    if (std::strcmp(key, "held_pool_bytes") == 0) {
        *value = (int64_t)device->freed.held_bytes();
        return FH_OK;
    }
    if (std::strcmp(key, "waiting_pool_bytes") == 0) {
        *value = (int64_t)device->freed.waiting_bytes();
        return FH_OK;
    }
    if (std::strcmp(key, "last_rows_plan") == 0) {
        *value = device->last_rows_plan;
        return FH_OK;
    }
    if (std::strcmp(key, "last_decoded_tile") == 0) {
        *value = device->last_decoded_tile;
        return FH_OK;
    }
    if (std::strcmp(key, "last_decoded_cut") == 0) {
        *value = device->last_decoded_cut;
        return FH_OK;
    }
    if (std::strcmp(key, "last_decoded_runs") == 0) {
        *value = device->last_decoded_runs;
        return FH_OK;
    }
    const int64_t* const setting = tuning_of(device, key);
    if (setting == nullptr) return fail(FH_ERR_PARAMETER, "unknown tuning key %s", key);
    *value = *setting;
    return FH_OK;
}

// ---- buffers -------------------------------------------------------------------

fh_status fh_buffer_alloc_uninitialized(fh_device* device, size_t bytes, fh_buffer** out) {
    if (device && device->capturing) return fail(FH_ERR_SYNCHRONIZATION, "not available while an execution is being recorded");
    if (device == nullptr || out == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    *out = nullptr;
    if (bytes == 0) return fail(FH_ERR_ALLOCATION, "zero-length buffer");
    FH_HIP(hipSetDevice(device->ordinal));
    void* p = nullptr;
    const size_t capacity = block_capacity(bytes);
    hipError_t e = take_block(device, capacity, &p);
    if (e != hipSuccess) return fail(FH_ERR_ALLOCATION, "hipMalloc(%zu): %s", capacity, hipGetErrorString(e));
    fh_buffer* b = new (std::nothrow) fh_buffer();
    if (b == nullptr) {
        (void)hipFree(p);
        return fail(FH_ERR_ALLOCATION, "out of host memory");
    }
    b->device = device;
    ++device->handles;
    b->ptr = p;
    b->bytes = bytes;
    b->capacity = capacity;
    *out = b;
    return FH_OK;
}

fh_status fh_buffer_alloc(fh_device* device, size_t bytes, fh_buffer** out) {
    fh_status st = fh_buffer_alloc_uninitialized(device, bytes, out);
    if (st != FH_OK) return st;
    const hipError_t e = hipMemsetAsync((*out)->ptr, 0, bytes, device->stream);
    if (e != hipSuccess) {
        fh_buffer_free(*out);
        *out = nullptr;
        return hip_fail(e, "hipMemsetAsync");
    }
    return FH_OK;
}

void fh_buffer_free(fh_buffer* buffer) {
    if (buffer == nullptr) return;
    fh_device* const d = buffer->device;
    if (!keep_block(d, *buffer)) release_memory(d, buffer->ptr);
    drop_device_handle(d);
    delete buffer;
}

size_t fh_buffer_size(const fh_buffer* buffer) { return buffer ? buffer->bytes : 0; }
void* fh_buffer_device_ptr(fh_buffer* buffer) {
    if (buffer == nullptr) return nullptr;
    buffer->exposed = true;
    return buffer->ptr;
}

fh_status fh_buffer_upload(fh_buffer* buffer, size_t offset, const void* src, size_t bytes) {
    if (buffer && buffer->device->capturing) return fail(FH_ERR_SYNCHRONIZATION, "not available while an execution is being recorded");
    if (buffer == nullptr || (src == nullptr && bytes)) return fail(FH_ERR_PARAMETER, "null argument");
    if (buffer->device->closed) return fail(FH_ERR_DEVICE_MISMATCH, "the buffer's device has been destroyed");
    if (offset > buffer->bytes || bytes > buffer->bytes - offset)
        return fail(FH_ERR_RANGE, "upload [%zu, +%zu) exceeds buffer of %zu bytes", offset, bytes,
                    buffer->bytes);
    if (bytes == 0) return FH_OK;
    hipStream_t s = buffer->device->stream;
    FH_HIP(hipMemcpyAsync(static_cast<uint8_t*>(buffer->ptr) + offset, src, bytes,
                          hipMemcpyHostToDevice, s));
    FH_HIP(hipStreamSynchronize(s));
    return FH_OK;
}

fh_status fh_buffer_download(const fh_buffer* buffer, size_t offset, void* dst, size_t bytes) {
    if (buffer && buffer->device->capturing) return fail(FH_ERR_SYNCHRONIZATION, "not available while an execution is being recorded");
    if (buffer == nullptr || (dst == nullptr && bytes)) return fail(FH_ERR_PARAMETER, "null argument");
    if (buffer->device->closed) return fail(FH_ERR_DEVICE_MISMATCH, "the buffer's device has been destroyed");
    if (offset > buffer->bytes || bytes > buffer->bytes - offset)
        return fail(FH_ERR_RANGE, "download [%zu, +%zu) exceeds buffer of %zu bytes", offset, bytes,
                    buffer->bytes);
    if (bytes == 0) return FH_OK;
    hipStream_t s = buffer->device->stream;
    hipError_t e = hipMemcpyAsync(dst, static_cast<const uint8_t*>(buffer->ptr) + offset, bytes,
                                  hipMemcpyDeviceToHost, s);
    if (e != hipSuccess) return hip_fail(e, "hipMemcpyAsync");
    e = hipStreamSynchronize(s);
    if (e != hipSuccess) return fail(FH_ERR_SYNCHRONIZATION, "stream: %s", hipGetErrorString(e));
    return FH_OK;
}

fh_status fh_buffer_fill_zero(fh_buffer* buffer, size_t offset, size_t bytes) {
    if (buffer && buffer->device->capturing) return fail(FH_ERR_SYNCHRONIZATION, "not available while an execution is being recorded");
    if (buffer == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (offset > buffer->bytes || bytes > buffer->bytes - offset)
        return fail(FH_ERR_RANGE, "fill exceeds buffer");
    if (bytes == 0) return FH_OK;
    FH_HIP(hipMemsetAsync(static_cast<uint8_t*>(buffer->ptr) + offset, 0, bytes,
                          buffer->device->stream));
    return FH_OK;
}

// ---- packed weights --------------------------------------------------------------

static bool f16_finite(const uint8_t* p) { return ((p[1] >> 2) & 0x1f) != 0x1f; }

fh_status fh_qmatrix_create(fh_device* device, uint32_t ggml_type, uint64_t rows, uint64_t cols,
                            uint64_t experts, const void* packed, size_t packed_len,
                            fh_qmatrix** out) {
    if (device && device->capturing) return fail(FH_ERR_SYNCHRONIZATION, "not available while an execution is being recorded");
    if (device == nullptr || out == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    *out = nullptr;
    const size_t bb = block_bytes(ggml_type);
    if (bb == 0) return fail(FH_ERR_GGUF, "unsupported quantized weight type %u", ggml_type);
    const char* name = ggml_type == kQ4K   ? "Q4_K"
                       : ggml_type == kQ5K ? "Q5_K"
                       : ggml_type == kQ6K ? "Q6_K"
                       : ggml_type == kQ8_0 ? "Q8_0"
                                            : "IQ4_XS";
    // a row is whole blocks: super-blocks of 256 weights, or for Q8_0 the 32-weight blocks of its GGML
    // geometry (src/loader/gguf.rs:99)
    const uint64_t unit = ggml_type == kQ8_0 ? 32 : 256;
    const size_t unit_bytes = ggml_type == kQ8_0 ? 34 : bb;
    if (rows == 0 || cols == 0 || cols % unit != 0)
        return fail(FH_ERR_SHAPE, "%s matrix requires nonempty rows and columns divisible by block size %u",
                    name, (unsigned)unit);
    if (experts == 0) return fail(FH_ERR_SHAPE, "quantized expert matrix row geometry mismatch");
    const uint64_t stored_cols = (cols + 255) / 256 * 256;
    unsigned __int128 total_rows = (unsigned __int128)rows * experts;
    unsigned __int128 byte_len = total_rows * (cols / unit) * unit_bytes;
    unsigned __int128 stored_len = total_rows * (stored_cols / 256) * bb;
    if (total_rows > 0xffffffffull || stored_len > (unsigned __int128)SIZE_MAX / 2)
        return fail(FH_ERR_SHAPE, "packed matrix byte size overflow");
    if (packed == nullptr) return fail(FH_ERR_PARAMETER, "null payload");
    if (packed_len % unit_bytes != 0)
        return fail(FH_ERR_GGUF, "tensor %s stream ended inside a block", name);
    if ((unsigned __int128)packed_len != byte_len)
        return fail(FH_ERR_SHAPE, "%s payload is %zu bytes, geometry needs %llu", name, packed_len,
                    (unsigned long long)byte_len);
    const uint8_t* p = static_cast<const uint8_t*>(packed);
    for (size_t off = 0; off < packed_len; off += unit_bytes) {
        bool ok = ggml_type == kQ6K     ? f16_finite(p + off + 208)
                  : ggml_type == kIQ4XS || ggml_type == kQ8_0 ? f16_finite(p + off)
                                        : (f16_finite(p + off) && f16_finite(p + off + 2));
        if (!ok) return fail(FH_ERR_WEIGHT, "%s scale must be finite", name);
    }
    // Q8_0 rows that do not end on a run of eight blocks are stored with the run completed by
    // empty blocks (scale and quants zero): the kernels then see rows of `stored_cols` weights,
    // and the entry points bring the activations to that width (pad_activations below)
    std::vector<uint8_t> staged;
    const size_t upload_len = (size_t)stored_len;
    if (stored_cols != cols) {
        try {
            staged.assign(upload_len, 0);
        } catch (const std::bad_alloc&) {
            return fail(FH_ERR_ALLOCATION, "out of host memory");
        }
        const size_t row_bytes = (size_t)(cols / 32) * 34, stored_row_bytes = (size_t)(stored_cols / 32) * 34;
        for (size_t r = 0; r < (size_t)total_rows; ++r)
            std::memcpy(staged.data() + r * stored_row_bytes, p + r * row_bytes, row_bytes);
        p = staged.data();
    }
    FH_HIP(hipSetDevice(device->ordinal));
    void* dptr = nullptr;
    // 16 spare bytes keep vector loads of the last block inside the allocation
    hipError_t e = allocate(device, &dptr, upload_len + 16);
    if (e != hipSuccess)
        return fail(FH_ERR_ALLOCATION, "hipMalloc(%zu): %s", upload_len, hipGetErrorString(e));
    e = hipMemcpyAsync(dptr, p, upload_len, hipMemcpyHostToDevice, device->stream);
    if (e == hipSuccess) e = hipMemsetAsync(static_cast<uint8_t*>(dptr) + upload_len, 0, 16, device->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(device->stream);
    if (e != hipSuccess) {
        (void)hipFree(dptr);
        return hip_fail(e, "weight upload");
    }
    fh_qmatrix* m = new (std::nothrow) fh_qmatrix();
    if (m == nullptr) {
        (void)hipFree(dptr);
        return fail(FH_ERR_ALLOCATION, "out of host memory");
    }
    m->device = device;
    ++device->handles;
    m->ptr = dptr;
    m->bytes = packed_len;
    m->ggml_type = ggml_type;
    m->rows = rows;
    m->cols = cols;
    m->stored_cols = stored_cols;
    m->experts = experts;
    *out = m;
    return FH_OK;
}

void fh_qmatrix_destroy(fh_qmatrix* matrix) {
    if (matrix == nullptr) return;
    release_memory(matrix->device, matrix->ptr);
    drop_device_handle(matrix->device);
    delete matrix;
}

uint64_t fh_qmatrix_rows(const fh_qmatrix* m) { return m ? m->rows : 0; }
uint64_t fh_qmatrix_columns(const fh_qmatrix* m) { return m ? m->cols : 0; }
uint64_t fh_qmatrix_experts(const fh_qmatrix* m) { return m ? m->experts : 0; }
uint32_t fh_qmatrix_ggml_type(const fh_qmatrix* m) { return m ? m->ggml_type : 0; }
size_t fh_qmatrix_byte_size(const fh_qmatrix* m) { return m ? m->bytes : 0; }
void* fh_qmatrix_device_ptr(fh_qmatrix* m) { return m ? m->ptr : nullptr; }

fh_status fh_dequantize(fh_device* device, const fh_qmatrix* weight, const fh_view* out) {
    if (device == nullptr || weight == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (weight->device != device) return fail(FH_ERR_DEVICE_MISMATCH, "weight belongs to another device");
    const uint64_t rows = weight->rows * weight->experts;
    Range o;
    fh_status st = resolve(device, out, rows * weight->cols, "dequantize output", &o);
    if (st != FH_OK) return st;
    device->last_operation = launch_dequantize(device->stream, weight->ggml_type, weight->ptr, rows, weight->stored_cols,
                                               weight->cols, const_cast<uint8_t*>(o.begin), out->dtype);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

fh_status fh_embedding_gather_quantized(fh_device* device, const fh_qmatrix* weight,
                                        const uint32_t* tokens, size_t count, const fh_view* out) {
    if (device && device->capturing) return fail(FH_ERR_SYNCHRONIZATION, "not available while an execution is being recorded");
    if (device == nullptr || weight == nullptr || (tokens == nullptr && count))
        return fail(FH_ERR_PARAMETER, "null argument");
    if (weight->device != device) return fail(FH_ERR_DEVICE_MISMATCH, "weight belongs to another device");
    const uint64_t rows = weight->rows * weight->experts;
    for (size_t i = 0; i < count; ++i)
        if (tokens[i] >= rows)
            return fail(FH_ERR_TOKEN, "token id %u is outside vocabulary of %llu", tokens[i],
                        (unsigned long long)rows);
    if (count == 0) return FH_OK;
    if (!fits_u32((uint64_t)count * weight->cols)) return fail(FH_ERR_SHAPE, "gather size overflow");
    Range o;
    fh_status st = resolve(device, out, (uint64_t)count * weight->cols, "gather output", &o);
    if (st != FH_OK) return st;
    // ids travel through the device scratch (the reference carries them in a tensor)
    size_t need = count * sizeof(uint32_t);
    fh_status sst = ensure_scratch(device, need);
    if (sst != FH_OK) return sst;
    FH_HIP(hipMemcpyAsync(scratch_data(device), tokens, need, hipMemcpyHostToDevice, device->stream));
    FH_HIP(hipStreamSynchronize(device->stream));
    device->last_operation =
        launch_embedding_gather(device->stream, weight->ggml_type, weight->ptr, weight->stored_cols, weight->cols,
                                reinterpret_cast<const uint32_t*>(scratch_data(device)), count,
                                const_cast<uint8_t*>(o.begin), out->dtype);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

// ---- dense projection --------------------------------------------------------------

namespace {

// A dense product's shape and the device's kernel switches; the caller sets w, x and y.
GemmArgs gemm_args(const fh_device* device, uint32_t ggml_type, uint64_t n, uint64_t k, uint32_t m, uint32_t x_dtype,
                   uint32_t y_dtype) {
    GemmArgs g{};
    g.ggml_type = ggml_type;
    g.n = (uint32_t)n;
    g.k = (uint32_t)k;
    g.m = m;
    g.x_dtype = x_dtype;
    g.y_dtype = y_dtype;
    g.cu_count = device->props.multiProcessorCount;
    g.wide_min_rows = (int)device->tuning.gemm_wide_min_rows;
    g.wide_shape = (int)device->tuning.gemm_wide_shape;
    g.wide32_tile = (int)device->tuning.gemm_wide32_tile;
    g.wide32_segments = (int)device->tuning.gemm_wide32_segments;
    g.decoded_min_rows = (int)device->tuning.gemm_decoded_min_rows;
    g.decoded_tile = (int)device->tuning.gemm_decoded_tile;
    g.decoded_segments = (int)device->tuning.gemm_decoded_segments;
    g.cut_tiles = true;
    g.skinny_max_rows = (int)device->tuning.gemm_skinny_max_rows;
    g.resident_switch = device->tuning.gemm_resident != 0;
    g.rows_resident = g.resident_switch && expert_rows_fit_lds((uint32_t)k, 1, 1);
    g.few_rows = device->tuning.gemm_few_tiles_split != 0;
    g.few_rows_always = device->tuning.gemm_few_tiles_split == 2;
    return g;
}

// Brings the scratch to what the product needs behind `used` bytes of the caller's at its head.  Partial sums
// only save time: where there is no room for them the product takes a kernel that needs fewer, at last one that
// needs none.
fh_status prepare_gemm(fh_device* device, GemmArgs& g, size_t used) {
    const size_t at = align256(used);
    fh_status st = FH_OK;
    for (;;) {
        const size_t partial_bytes = gemm_partial_bytes(g);
        st = partial_bytes != 0 ? optional_scratch(device, at + partial_bytes) : ensure_scratch(device, used);
        if (st != FH_ERR_ALLOCATION || partial_bytes == 0) break;
        if (g.decoded.runs != 0) {
            g.decoded.runs = 0;
        } else if (g.rows_plan.pairs) {
            g.rows_plan = g.rows_else;
            if (g.rows_plan.rows == 0) return ensure_scratch(device, used);
        } else if (g.rows_plan.rows != 0) {
            g.rows_plan = RowsPlan{};
            if (g.x_dtype == FH_F32) return ensure_scratch(device, used);   // no tile takes exact f32 rows
            if (!g.cut_tiles) g.few_rows = false;
        } else {
            g.cut_tiles = false;
            g.tile = TileChoice{};
            gemm_takes_rows(g);
        }
    }
    if (st != FH_OK) return st;
    g.counters = scratch_counters(device);
    g.partials = reinterpret_cast<float*>(scratch_data(device) + at);
    return FH_OK;
}

const char* run_gemm(fh_device* device, GemmArgs& g) {
    const RowsPlan& plan = g.rows_plan;
    device->last_rows_plan = plan.rows * 1000 + plan.tiles * 100 + plan.segments;
    const int64_t decoded_tile = g.decoded.runs != 0 ? g.decoded.run[0].tile : 0;
    device->last_decoded_tile = g.decoded.segments == 1 ? decoded_tile : 0;
    device->last_decoded_cut = g.decoded.segments == 2 ? decoded_tile : 0;
    device->last_decoded_runs = g.decoded.runs;
    return launch_gemm(device->stream, g);
}

// the exact product of several rows, by whichever kernel
const char* batch_name(uint32_t ggml_type) {
    return ggml_type == kQ4K    ? "q4_k_gemm"
           : ggml_type == kQ5K  ? "q5_k_gemm"
           : ggml_type == kQ6K  ? "q6_k_gemm"
           : ggml_type == kQ8_0 ? "q8_0_gemm"
                                : "iq4_xs_gemm";
}

// whether a dense GEMV of m plain rows runs on the streamed kernel
bool gemv_streams(const fh_device* device, uint32_t ggml_type, uint64_t n, uint64_t k, uint32_t m) {
    GemvArgs a{};
    a.ggml_type = ggml_type;
    a.n = (uint32_t)n;
    a.k = (uint32_t)k;
    a.m = m;
    a.cu_count = device->props.multiProcessorCount;
    a.stream = (int)device->tuning.gemv_stream;
    a.ksplit = (int)device->tuning.k_quant_gemv_ksplit;
    a.x_mode = kXPlain;
    StreamPlan plan;
    return gemv_takes_stream(a, &plan);
}

// `f32_tile_from`: row count from which f32 activations take the f16 tiles; negative = the
// device's gemm_f32_min_rows setting
fh_status project(fh_device* device, const fh_qmatrix* weight, const fh_view* x, uint32_t m,
                  const fh_view* y, bool silu_mul, int64_t f32_tile_from = -1) {
    if (device == nullptr || weight == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (weight->device != device) {
        g_last_error = "weight belongs to another device";
        return FH_ERR_DEVICE_MISMATCH;
    }
    const uint64_t n = weight->rows * weight->experts, k = weight->cols;
    if (m == 0 || k > 0xffffffffull - 32)
        return fail(FH_ERR_SHAPE, "quantized projection requires [M,K] matching [N,K]");
    if (weight->padded()) {
        const fh_qmatrix stored = as_stored(weight);
        PaddedActivations pad(device, weight);
        fh_view px{};
        pad.add(x, (uint64_t)m * (silu_mul ? 2 : 1), "projection input", &px);
        fh_status pst = pad.run();
        if (pst == FH_OK) pst = pad.keep_apart(y, (uint64_t)m * n, "projection output", "projection output aliases its input");
        if (pst != FH_OK) return pst;
        return project(device, &stored, &px, m, y, silu_mul, f32_tile_from);
    }
    const uint64_t x_elements = (uint64_t)m * k * (silu_mul ? 2 : 1);
    if (!fits_u32(x_elements) || !fits_u32((uint64_t)m * n) || !fits_u32(n))
        return fail(FH_ERR_SHAPE, "index does not fit in 32 bits");
    Range xr, yr;
    fh_status st = resolve(device, x, x_elements, "projection input", &xr);
    if (st != FH_OK) return st;
    st = resolve(device, y, (uint64_t)m * n, "projection output", &yr);
    if (st != FH_OK) return st;
    if (overlaps(xr, yr)) return fail(FH_ERR_RANGE, "projection output aliases its input");

    // f32 activations stay on exact f32 weights (the GEMV kernel, once per row) unless the
    // caller asks for the tile kernels from some row count on, as the reference's hybrid
    // engine does from 5 rows (HybridModel::project, src/hybrid/engine.rs:3407-3500): the
    // activations are then rounded to f16 into the device scratch first.
    const int64_t f32_tile_rows = f32_tile_from >= 0 ? f32_tile_from : device->tuning.gemm_f32_min_rows;
    const bool f32_tile = !silu_mul && x->dtype == FH_F32 && f32_tile_rows > 0 && m >= (uint64_t)f32_tile_rows &&
                          ((uintptr_t)xr.begin & 15u) == 0;
    const bool tile = f32_tile || (!silu_mul && m >= (uint32_t)device->tuning.gemm_min_rows && x->dtype != FH_F32);
    // A batch of exact f32 rows: the GEMV kernels read every weight once per row, the few-rows kernel
    // once per sixteen.  Against the FMA GEMV f32_rows_pay decides.  Where the streamed GEMV would run, the few-rows
    // kernel takes over from five Q4_K rows and four Q6_K rows on: it is the faster one from six (5 / 6 / 16 x 17408
    // x 5120 Q4_K 47.8 / 47.0 / 46.0 against 43.8 / 51.7 / 121 us, 5 / 6 x 4096 x 4096 11.8 / 11.7 against 11.1 / 12.4)
    // and at five the closer one to 64 bits (1e-7; the streamed kernel's operands are f16 pairs).  Where a GEMV
    // kernel or its K segments are asked for by name, those run.
    const bool f32_batch = !tile && !silu_mul && x->dtype == FH_F32 && m >= (weight->ggml_type == kQ4K ? 5u : 4u) &&
                           m >= (uint32_t)device->tuning.gemm_min_rows && device->tuning.gemv_stream == 1 &&
                           device->tuning.k_quant_gemv_ksplit == 0;
    device->last_rows_plan = device->last_decoded_tile = device->last_decoded_cut = device->last_decoded_runs = 0;
    GemmArgs g{};
    if (tile || f32_batch) g = gemm_args(device, weight->ggml_type, n, k, m, f32_tile ? FH_F16 : x->dtype, y->dtype);
    if (f32_batch && g.few_rows) {
        g.rows_plan = gemm_rows_plan(g.ggml_type, g.n, g.k, g.m, g.x_dtype, g.cu_count);
        if (g.rows_plan.counters > fh_device::kCounterWords || !rows_batch_fits(g.rows_plan, g.k, g.x_dtype) ||
            (!g.few_rows_always && !gemv_streams(device, weight->ggml_type, n, k, m) &&
             !f32_rows_pay(g.rows_plan, g.ggml_type, g.n, g.k, m, g.cu_count)))
            g.rows_plan = RowsPlan{};
        if (!g.few_rows_always && pairs_pay(g.ggml_type, g.n, g.k, m) && ((uintptr_t)xr.begin & 15u) == 0) {
            g.rows_else = g.rows_plan;
            g.rows_plan = gemm_pairs_plan(g.n, g.k, g.m, g.cu_count);
        }
    }
    if (tile && !gemm_takes_rows(g)) gemm_takes_decoded(g);
    if (tile || g.rows_plan.rows != 0) {
        st = prepare_gemm(device, g, f32_tile ? (size_t)m * k * sizeof(uint16_t) : 0);
        if (st != FH_OK) return st;
    }
    if (tile || g.rows_plan.rows != 0) {
        g.w = weight->ptr;
        g.x = xr.begin;
        g.y = const_cast<uint8_t*>(yr.begin);
        if (f32_tile) {
            launch_round_to_f16(device->stream, reinterpret_cast<const float*>(xr.begin),
                                reinterpret_cast<uint16_t*>(scratch_data(device)), (size_t)m * k);
            g.x = scratch_data(device);
        }
        const char* const name = run_gemm(device, g);
        device->last_operation = tile ? name : batch_name(weight->ggml_type);
    } else {
        GemvArgs a{};
        a.ggml_type = weight->ggml_type;
        a.w = weight->ptr;
        a.x = xr.begin;
        a.y = const_cast<uint8_t*>(yr.begin);
        a.n = (uint32_t)n;
        a.k = (uint32_t)k;
        a.m = m;
        a.x_dtype = x->dtype;
        a.y_dtype = y->dtype;
        a.metadata = nullptr;
        a.experts = 1;
        a.ksplit = (int)device->tuning.k_quant_gemv_ksplit;
        a.stream = (int)device->tuning.gemv_stream;
        a.stream_own = device->tuning.gemv_stream_own_loads != 0;
        a.ring = (int)device->tuning.gemv_ring;
        a.cu_count = device->props.multiProcessorCount;
        a.x_mode = silu_mul ? kXSiluMul : kXPlain;
        a.x_rows = m;
        // One activated row stays on the FMA kernel: the streamed Q4_K one's operands are f16 pairs and the matrix core
        // keeps few bits of a subnormal weight (rel-L2 to 64 bits 2e-6 to 1.4e-5 on rows of mean weights, against 1.0e-7
        // to 2.0e-7).  The streamed Q6_K kernel sums integers and is the closer one for f32 rows (1.0e-7 against
        // 2.0e-7; 16-bit rows 0.95e-7 on either): they take it from 200,000 super-blocks on.  us with the activation, weights
        // out of every cache, FMA / streamed: 2048 x 28672 22.3 / 21.9, 4096 x 12800 22.7 / 20.5, 4096 x 14336 23.3 / 20.7, 5120 x
        // 17408 29.2 / 26.7, 4096 x 28672 36.0 / 34.0, 8192 x 14336 37.8 / 31.6; below, the longest rows gain nothing
        // (1024 x 28672 16.6 / 16.8, 1250 x 17408 13.9 / 13.9), shorter ones up to a seventh (3000 x 12800 19.6 / 16.7).
        // Activating in place, every workgroup activates the whole row again;
        // for large matrices the row is written out first, as the separate expert_silu_mul would, with the same
        // bits.  us, in place against written first: 5120 x 17408 26.5 / 20.6 (Q6_K 36.2 / 28.2), 5120 x 5120
        // 10.8 / 10.0 (15.3 / 13.1), 2048 x 12800 12.3 / 11.8 (16.1 / 14.7); 4096 x 4096, where the second launch
        // costs more, 8.3 / 9.4 (9.3 / 9.6).
        if (silu_mul && m == 1 && (weight->ggml_type == kQ4K || weight->ggml_type == kQ6K) && n * (k / 256) >= 81920u) {
            GemvArgs plain = a;
            plain.x_mode = kXPlain;
            if (weight->ggml_type != kQ6K || x->dtype != FH_F32 || n * (k / 256) < 200000u) plain.stream = 0;
            auto partials_of = [&] { return align256((size_t)gemv_scratch(plain).segments * n * sizeof(float)); };
            if (!scratch_available(device, partials_of() + (size_t)k * dtype_bytes(x->dtype))) plain.stream = 0;   // fewer segments
            const size_t partial_bytes = partials_of();
            const size_t bytes = partial_bytes + (size_t)k * dtype_bytes(x->dtype);
            if (scratch_available(device, bytes)) {
                st = ensure_scratch(device, bytes);
                if (st != FH_OK) return st;
                uint8_t* const row = scratch_data(device) + partial_bytes;   // behind the partial sums
                launch_expert_silu_mul(device->stream, xr.begin, row, 1, (uint32_t)k, x->dtype, x->dtype);
                plain.x = row;
                a = plain;
            }
        }
        const char* name = "";
        st = run_gemv(device, a, &name);
        if (st != FH_OK) return st;
        device->last_operation = m > 1 ? batch_name(weight->ggml_type) : name;
    }
    FH_HIP(hipGetLastError());
    return FH_OK;
}

}  // namespace

fh_status fh_project_quantized(fh_device* device, const fh_qmatrix* weight, const fh_view* x,
                               uint32_t m, const fh_view* y) {
    return project(device, weight, x, m, y, false);
}

fh_status fh_project_silu_mul_quantized(fh_device* device, const fh_qmatrix* weight, const fh_view* packed,
                                        uint32_t m, const fh_view* y) {
    return project(device, weight, packed, m, y, true);
}

// fh_project_quantized through the per-row GEMV kernels only, with the kernel's scratch in the
// library's fixed array: no hipMalloc, hipFree or synchronisation on any path.
fh_status fh_project_quantized_no_alloc(fh_device* device, const fh_qmatrix* weight, const fh_view* x,
                                        uint32_t m, const fh_view* y) {
    if (device == nullptr || weight == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (weight->device != device) return fail(FH_ERR_DEVICE_MISMATCH, "weight belongs to another device");
    if (device->fixed_scratch == nullptr) return fail(FH_ERR_DISPATCH, "the fixed scratch is not set up");
    if (weight->padded())
        return fail(FH_ERR_SHAPE, "rows of %llu weights are stored padded and need a temporary for the activations: "
                    "fh_project_quantized takes them", (unsigned long long)weight->cols);
    const uint64_t n = weight->rows * weight->experts, k = weight->cols;
    if (m == 0 || k > 0xffffffffull - 32)
        return fail(FH_ERR_SHAPE, "quantized projection requires [M,K] matching [N,K]");
    if (!fits_u32((uint64_t)m * k) || !fits_u32((uint64_t)m * n) || !fits_u32(n) || m > 65535u)
        return fail(FH_ERR_SHAPE, "index does not fit in 32 bits");
    Range xr, yr;
    fh_status st = resolve(device, x, (uint64_t)m * k, "projection input", &xr);
    if (st != FH_OK) return st;
    st = resolve(device, y, (uint64_t)m * n, "projection output", &yr);
    if (st != FH_OK) return st;
    if (overlaps(xr, yr)) return fail(FH_ERR_RANGE, "projection output aliases its input");
    GemvArgs a{};
    a.ggml_type = weight->ggml_type;
    a.w = weight->ptr;
    a.x = xr.begin;
    a.y = const_cast<uint8_t*>(yr.begin);
    a.n = (uint32_t)n;
    a.k = (uint32_t)k;
    a.m = m;
    a.x_dtype = x->dtype;
    a.y_dtype = y->dtype;
    a.experts = 1;
    a.ksplit = (int)device->tuning.k_quant_gemv_ksplit;
    a.stream = (int)device->tuning.gemv_stream;
    a.stream_own = device->tuning.gemv_stream_own_loads != 0;
    a.ring = (int)device->tuning.gemv_ring;
    a.cu_count = device->props.multiProcessorCount;
    a.x_mode = kXPlain;
    a.x_rows = m;
    GemvScratch plan = gemv_scratch(a);
    if (a.ring != 0 && (uint64_t)plan.segments * m * n * sizeof(float) > kFixedScratchBytes - kFixedCounterWords * sizeof(uint32_t)) {
        a.ring = 0;   // its segments may be more than the fixed scratch has room for
        plan = gemv_scratch(a);
    }
    if (plan.segments > 1) {
        const uint64_t counters = (uint64_t)plan.tiles * m;
        const uint64_t partial_bytes = (uint64_t)plan.segments * m * n * sizeof(float);
        if (counters > kFixedCounterWords || partial_bytes > kFixedScratchBytes - kFixedCounterWords * sizeof(uint32_t))
            return fail(FH_ERR_SHAPE,
                        "projection needs %llu counters and %llu bytes of partial sums; the fixed scratch holds %zu and %zu",
                        (unsigned long long)counters, (unsigned long long)partial_bytes, kFixedCounterWords,
                        kFixedScratchBytes - kFixedCounterWords * sizeof(uint32_t));
        uint8_t* const base = static_cast<uint8_t*>(device->fixed_scratch);
        a.counters = reinterpret_cast<uint32_t*>(base);
        a.partials = reinterpret_cast<float*>(base + kFixedCounterWords * sizeof(uint32_t));
    }
    device->last_operation = launch_gemv(device->stream, a, plan);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

// ---- measurement ----------------------------------------------------------------------

fh_status fh_probe_read(fh_device* device, const fh_qmatrix* weight) {
    if (device == nullptr || weight == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (weight->device != device) return fail(FH_ERR_PARAMETER, "matrix belongs to another device");
    fh_status st = ensure_scratch(device, 0);
    if (st != FH_OK) return st;
    device->last_operation = launch_read_probe(device->stream, weight->ptr, weight->bytes,
                                               reinterpret_cast<uint32_t*>(scratch_data(device)), device->tuning.probe_read_form);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

fh_status fh_probe_mfma(fh_device* device, uint32_t shape, uint32_t groups, uint32_t iterations, double* flops) {
    if (device == nullptr || flops == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (shape > 2 || groups == 0 || groups > 65535 || iterations == 0)
        return fail(FH_ERR_SHAPE, "mfma probe: shape 0, 1 or 2, 1..65535 workgroups, at least one iteration");
    fh_status st = ensure_scratch(device, (size_t)groups * 256 * sizeof(float));
    if (st != FH_OK) return st;
    device->last_operation = launch_mfma_probe(device->stream, (int)shape, groups, iterations,
                                               reinterpret_cast<float*>(scratch_data(device)), flops);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

fh_status fh_probe_coissue(fh_device* device, uint32_t groups, uint32_t iterations, uint32_t mfma,
                           uint32_t valu_rounds) {
    if (device == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (groups == 0 || groups > 65535 || iterations == 0 || (mfma == 0 && valu_rounds == 0))
        return fail(FH_ERR_SHAPE, "co-issue probe: 1..65535 workgroups, at least one iteration, something to run");
    fh_status st = ensure_scratch(device, (size_t)groups * 512 * sizeof(float));
    if (st != FH_OK) return st;
    device->last_operation = launch_coissue_probe(device->stream, groups, iterations, mfma, valu_rounds,
                                                  reinterpret_cast<float*>(scratch_data(device)));
    FH_HIP(hipGetLastError());
    return FH_OK;
}

// ---- mixture of experts -------------------------------------------------------------

fh_status fh_argmax_rows(fh_device* device, const fh_view* logits, uint32_t rows, uint32_t width,
                         const fh_view* out) {
    if (device == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (rows == 0 || width == 0 || !fits_u32((uint64_t)rows * width))
        return fail(FH_ERR_SHAPE, "argmax requires nonempty [rows,width]");
    if (out == nullptr || out->dtype != FH_F32) return fail(FH_ERR_DTYPE, "argmax output is an f32 carrier of [rows,2]");
    Range lr, orr;
    fh_status st = resolve(device, logits, (uint64_t)rows * width, "argmax input", &lr);
    if (st != FH_OK) return st;
    st = resolve(device, out, (uint64_t)rows * 2, "argmax output", &orr, 4);
    if (st != FH_OK) return st;
    if (overlaps(lr, orr)) return fail(FH_ERR_RANGE, "argmax output aliases its input");
    st = ensure_scratch(device, argmax_partial_bytes(rows, width));   // 9 MiB at most, which it always holds
    if (st != FH_OK) return st;
    device->last_operation = launch_argmax_rows(device->stream, lr.begin, logits->dtype, rows, width,
                                                scratch_data(device), scratch_counters(device),
                                                reinterpret_cast<uint32_t*>(const_cast<uint8_t*>(orr.begin)));
    FH_HIP(hipGetLastError());
    return FH_OK;
}

fh_status fh_add_rmsnorm(fh_device* device, const fh_view* a, const fh_view* b, const fh_view* weight,
                         uint32_t rows, uint32_t width, float epsilon, const fh_view* residual,
                         const fh_view* normed) {
    if (device == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (rows == 0 || width == 0 || width > 0xffffffffu - 256u || !fits_u32((uint64_t)rows * width))
        return fail(FH_ERR_SHAPE, "fused add+RMSNorm requires nonempty [rows,width]");
    if (a == nullptr || b == nullptr || weight == nullptr || residual == nullptr || normed == nullptr)
        return fail(FH_ERR_RANGE, "fused add+RMSNorm: null view");
    if (a->dtype != b->dtype || weight->dtype != a->dtype || residual->dtype != a->dtype || normed->dtype != a->dtype)
        return fail(FH_ERR_SHAPE, "fused add+RMSNorm operands must match");
    if (!std::isfinite(epsilon) || epsilon <= 0.f)
        return fail(FH_ERR_PARAMETER, "epsilon must be finite and positive");
    const uint64_t count = (uint64_t)rows * width;
    Range ar, br, wr, rr, nr;
    fh_status st = resolve(device, a, count, "add+RMSNorm a", &ar);
    if (st != FH_OK) return st;
    if ((st = resolve(device, b, count, "add+RMSNorm b", &br)) != FH_OK) return st;
    if ((st = resolve(device, weight, width, "add+RMSNorm weight", &wr)) != FH_OK) return st;
    if ((st = resolve(device, residual, count, "add+RMSNorm residual", &rr)) != FH_OK) return st;
    if ((st = resolve(device, normed, count, "add+RMSNorm output", &nr)) != FH_OK) return st;
    for (const Range* out : {&rr, &nr}) {
        if (overlaps(*out, ar) || overlaps(*out, br) || overlaps(*out, wr))
            return fail(FH_ERR_RANGE, "add+RMSNorm outputs alias an operand");
    }
    if (overlaps(rr, nr)) return fail(FH_ERR_RANGE, "add+RMSNorm outputs alias each other");
    device->last_operation = launch_add_rmsnorm(device->stream, ar.begin, br.begin, wr.begin,
                                                const_cast<uint8_t*>(rr.begin), const_cast<uint8_t*>(nr.begin), rows,
                                                width, a->dtype, epsilon);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

namespace {

fh_status route(fh_device* device, const fh_view* logits, uint32_t tokens, const fh_view* selection_bias,
                const fh_routing_policy* policy, const fh_view* metadata, bool ranked, const fh_view* gate_x,
                const fh_view* gate_w, uint32_t hidden, const fh_view* shared_gate, const fh_view* ids = nullptr,
                const fh_view* weights = nullptr, RouteTokenArgs* defer = nullptr) {
    if (device == nullptr || policy == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    const fh_routing_policy& p = *policy;
    if (tokens == 0 || p.experts == 0 || p.top_k == 0 || p.top_k > 16 || p.top_k > p.experts ||
        !std::isfinite(p.normalization_epsilon) || p.normalization_epsilon < 0.f ||
        !std::isfinite(p.routed_scaling_factor) || p.routed_scaling_factor <= 0.f)
        return fail(FH_ERR_SHAPE, "invalid sparse routing geometry");
    if (p.experts > 1024) return fail(FH_ERR_SHAPE, "routing supports at most 1024 experts");
    if (!fits_u32((uint64_t)tokens * p.top_k * 3) || !fits_u32((uint64_t)tokens * p.experts))
        return fail(FH_ERR_SHAPE, "expert assignment count overflow");
    Range lr, mr, br{nullptr, 0};
    // the kernel loads logits one element at a time: a chunk of 16-bit logits over an odd number of experts
    // may start at any element
    fh_status st = resolve(device, logits, (uint64_t)tokens * p.experts, "router logits", &lr,
                           logits != nullptr ? dtype_bytes(logits->dtype) : 4);
    if (st != FH_OK) return st == FH_ERR_DEVICE_MISMATCH ? fail(FH_ERR_SHAPE, "invalid sparse routing geometry") : st;
    if (selection_bias != nullptr) {
        if (selection_bias->dtype != FH_F32) return fail(FH_ERR_SHAPE, "invalid sparse routing geometry");
        st = resolve(device, selection_bias, p.experts, "selection bias", &br, 4);
        if (st != FH_OK) return st == FH_ERR_DEVICE_MISMATCH ? fail(FH_ERR_SHAPE, "invalid sparse routing geometry") : st;
    }
    RouteExtras extras;
    extras.rank_order = ranked ? 1u : 0u;
    mr = Range{nullptr, 0};
    if (ids == nullptr) {
        if (metadata == nullptr || metadata->dtype != FH_F32)
            return fail(FH_ERR_DTYPE, "routing metadata must be f32");
        st = resolve(device, metadata, (uint64_t)tokens * p.top_k * 3, "routing metadata", &mr, 4);
        if (st != FH_OK) return st;
        if (overlaps(lr, mr)) return fail(FH_ERR_RANGE, "routing metadata aliases the logits");
    } else {
        // the hybrid engine's layout: ids and weights as two [tokens, top_k] f32 carriers
        if (weights == nullptr || ids->dtype != FH_F32 || weights->dtype != FH_F32)
            return fail(FH_ERR_DTYPE, "route ids and weights are f32 carriers");
        Range ir, wr;
        st = resolve(device, ids, (uint64_t)tokens * p.top_k, "route ids", &ir, 4);
        if (st != FH_OK) return st;
        st = resolve(device, weights, (uint64_t)tokens * p.top_k, "route weights", &wr, 4);
        if (st != FH_OK) return st;
        if (overlaps(lr, ir) || overlaps(lr, wr) || overlaps(ir, wr))
            return fail(FH_ERR_RANGE, "route outputs alias the logits or each other");
        extras.ids_out = reinterpret_cast<float*>(const_cast<uint8_t*>(ir.begin));
        extras.weights_out = reinterpret_cast<float*>(const_cast<uint8_t*>(wr.begin));
    }
    if (shared_gate != nullptr) {
        if (shared_gate->dtype != FH_F32) return fail(FH_ERR_DTYPE, "the shared-expert gate is f32");
        Range gr;
        st = resolve(device, shared_gate, tokens, "shared-expert gate", &gr, 4);
        if (st != FH_OK) return st;
        extras.shared_gate = reinterpret_cast<float*>(const_cast<uint8_t*>(gr.begin));
        if (gate_w != nullptr) {
            if (gate_w->dtype != FH_F32 || gate_x == nullptr || hidden == 0 || !fits_u32((uint64_t)tokens * hidden))
                return fail(FH_ERR_SHAPE, "the shared-expert gate needs x [tokens, hidden] and an f32 vector [hidden]");
            Range xr, wr;
            st = resolve(device, gate_x, (uint64_t)tokens * hidden, "gate activations", &xr);
            if (st != FH_OK) return st;
            st = resolve(device, gate_w, hidden, "gate vector", &wr, 4);
            if (st != FH_OK) return st;
            extras.gate_x = xr.begin;
            extras.gate_x_dtype = gate_x->dtype;
            extras.gate_w = reinterpret_cast<const float*>(wr.begin);
            extras.hidden = hidden;
        }
    }
    if (defer != nullptr) {
        // checked as a launch would be; the projection that follows routes the token itself
        RouteTokenArgs& r = *defer;
        r = RouteTokenArgs{};
        r.logits = lr.begin;
        r.logits_dtype = logits->dtype;
        r.bias = reinterpret_cast<const float*>(br.begin);
        r.metadata = reinterpret_cast<float*>(const_cast<uint8_t*>(mr.begin));
        r.experts = p.experts;
        r.top_k = p.top_k;
        r.sigmoid = p.sigmoid;
        r.normalize = p.normalize_top_k_prob;
        r.eps = p.normalization_epsilon;
        r.scaling = p.routed_scaling_factor;
        r.rank_order = extras.rank_order;
        return FH_OK;
    }
    device->last_operation = launch_moe_route(
        device->stream, lr.begin, logits->dtype, reinterpret_cast<const float*>(br.begin),
        reinterpret_cast<float*>(const_cast<uint8_t*>(mr.begin)), tokens, p, extras);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

}  // namespace

fh_status fh_moe_route(fh_device* device, const fh_view* logits, uint32_t tokens,
                       const fh_view* selection_bias, const fh_routing_policy* policy,
                       const fh_view* metadata) {
    return route(device, logits, tokens, selection_bias, policy, metadata, false, nullptr, nullptr, 0, nullptr);
}

fh_status fh_moe_route_ranked(fh_device* device, const fh_view* logits, uint32_t tokens,
                              const fh_routing_policy* policy, const fh_view* x, const fh_view* gate_vector,
                              uint32_t hidden, const fh_view* metadata, const fh_view* shared_gate) {
    return route(device, logits, tokens, nullptr, policy, metadata, true, x, gate_vector, hidden, shared_gate);
}

// ---- the hybrid engine's MoE stages over plain id / weight arrays ----------------------

fh_status fh_hybrid_moe_route(fh_device* device, const fh_view* logits, uint32_t tokens,
                              const fh_routing_policy* policy, const fh_view* x, const fh_view* gate_vector,
                              uint32_t hidden, const fh_view* ids, const fh_view* weights,
                              const fh_view* shared_gate) {
    if (ids == nullptr) return fail(FH_ERR_RANGE, "route ids: null view");
    return route(device, logits, tokens, nullptr, policy, nullptr, true, x, gate_vector, hidden, shared_gate, ids,
                 weights);
}

fh_status fh_hybrid_project(fh_device* device, const fh_qmatrix* weight, const fh_view* x, uint32_t m,
                            const fh_view* y, uint32_t exact) {
    // HybridModel::project (src/hybrid/engine.rs:3407-3500): one row and `exact` keep f32
    // weights; 2..4 rows are a batched GEMV, also exact; from 5 rows (MVB_MAX_ROWS + 1,
    // :3584) the rows go through f16 tiles
    const fh_status st = project(device, weight, x, m, y, false, exact ? 0 : 5);
    if (st != FH_OK) return st;
    static const char* const names[4][5] = {
        {"h_mv_q4_k", "h_mv_q5_k", "h_mv_q6_k", "h_mv_q8_0", "h_mv_iq4_xs"},
        {"h_mvb_q4_k", "h_mvb_q5_k", "h_mvb_q6_k", "h_mvb_q8_0", "h_mvb_iq4_xs"},
        {"h_mms_q4_k", "h_mms_q5_k", "h_mms_q6_k", "h_mms_q8_0", "h_mms_iq4_xs"},
        {"h_mm_q4_k", "h_mm_q5_k", "h_mm_q6_k", "h_mm_q8_0", "h_mm_iq4_xs"}};
    const int tier = m == 1 || exact ? 0 : m <= 4 ? 1 : m <= 32 ? 2 : 3;
    const int f = weight->ggml_type == kQ4K ? 0 : weight->ggml_type == kQ5K ? 1 : weight->ggml_type == kQ6K ? 2
                  : weight->ggml_type == kQ8_0 ? 3 : 4;
    device->last_operation = names[tier][f];
    return FH_OK;
}

namespace {

// A shared expert (dense [rows, k] matrix every token also runs) can ride in a routed
// launch: tokens entries more, reading the token rows or rows of its own (x), writing y.
struct SharedExpert {
    const fh_qmatrix* weight = nullptr;
    uint32_t tokens = 0;
    const fh_view* x = nullptr;
    const fh_view* y = nullptr;
};

// The shared expert of a launch on a padded matrix: its matrix as stored, its own activations padded too.
// `parts`: runs of `cols` elements per row of the shared expert's input.
struct PaddedRider {
    fh_qmatrix stored{};
    fh_view x{};
    SharedExpert rider;
    const SharedExpert* get(const SharedExpert* shared) const { return shared != nullptr ? &rider : nullptr; }
};

fh_status pad_rider(PaddedActivations& pad, const fh_qmatrix* weight, const SharedExpert* shared, uint32_t parts,
                    PaddedRider* out) {
    if (shared == nullptr) return FH_OK;
    if (shared->weight == nullptr || shared->y == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (shared->weight->cols != weight->cols)
        return fail(FH_ERR_SHAPE, "the shared expert's matrix must have one expert's shape and format");
    out->stored = as_stored(shared->weight);
    out->rider = *shared;
    out->rider.weight = &out->stored;
    if (shared->x != nullptr) {
        pad.add(shared->x, (uint64_t)shared->tokens * parts, "shared expert input", &out->x);
        out->rider.x = &out->x;
    }
    return FH_OK;
}

fh_status hybrid_project_id(fh_device* device, const fh_qmatrix* weight, const fh_view* x, const fh_view* ids,
                            uint32_t routes, uint32_t x_div, const fh_view* y, const SharedExpert* shared) {
    if (device == nullptr || weight == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (weight->device != device || routes == 0 || x_div == 0 || routes % x_div != 0 || ids == nullptr ||
        ids->dtype != FH_F32)
        return fail(FH_ERR_SHAPE, "expert projection geometry");
    if (weight->padded()) {
        const fh_qmatrix stored = as_stored(weight);
        PaddedActivations pad(device, weight);
        PaddedRider pr;
        fh_view px{};
        pad.add(x, (uint64_t)routes / x_div, "expert input", &px);
        fh_status pst = pad_rider(pad, weight, shared, 1, &pr);
        if (pst == FH_OK) pst = pad.run();
        if (pst == FH_OK) pst = pad.keep_apart(y, (uint64_t)routes * weight->rows, "expert output", "expert output aliases an input");
        if (pst == FH_OK && shared != nullptr)
            pst = pad.keep_apart(shared->y, (uint64_t)shared->tokens * weight->rows, "shared expert output",
                                 "shared expert output aliases another tensor");
        if (pst != FH_OK) return pst;
        return hybrid_project_id(device, &stored, &px, ids, routes, x_div, y, pr.get(shared));
    }
    const uint64_t rows = weight->rows, k = weight->cols;
    if (!fits_u32((uint64_t)routes * rows) || !fits_u32((uint64_t)routes / x_div * k))
        return fail(FH_ERR_SHAPE, "index does not fit in 32 bits");
    Range xr, ir, yr;
    fh_status st = resolve(device, x, (uint64_t)routes / x_div * k, "expert input", &xr);
    if (st != FH_OK) return st;
    st = resolve(device, ids, routes, "route ids", &ir, 4);
    if (st != FH_OK) return st;
    st = resolve(device, y, (uint64_t)routes * rows, "expert output", &yr);
    if (st != FH_OK) return st;
    if (overlaps(xr, yr) || overlaps(ir, yr)) return fail(FH_ERR_RANGE, "expert output aliases an input");
    Range sxr{nullptr, 0}, syr{nullptr, 0};
    if (shared != nullptr) {
        const fh_qmatrix* sw = shared->weight;
        if (sw == nullptr || shared->y == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
        if (sw->device != device) {
            g_last_error = "weight belongs to another device";
            return FH_ERR_DEVICE_MISMATCH;
        }
        if (sw->experts != 1 || sw->rows != rows || sw->cols != k || sw->ggml_type != weight->ggml_type)
            return fail(FH_ERR_SHAPE, "the shared expert's matrix must have one expert's shape and format");
        // without rows of its own the shared expert reads the token rows of x, one per x_div routes
        if (shared->tokens == 0 || (shared->x == nullptr && shared->tokens != routes / x_div) ||
            !fits_u32((uint64_t)routes + shared->tokens) || !fits_u32((uint64_t)shared->tokens * rows) ||
            !fits_u32((uint64_t)shared->tokens * k))
            return fail(FH_ERR_SHAPE, "the shared expert runs once per token");
        if (shared->y->dtype != y->dtype || (shared->x != nullptr && shared->x->dtype != x->dtype))
            return fail(FH_ERR_DTYPE, "the shared expert's tensors differ in dtype from the routed ones");
        st = resolve(device, shared->y, (uint64_t)shared->tokens * rows, "shared expert output", &syr);
        if (st != FH_OK) return st;
        if (shared->x != nullptr) {
            st = resolve(device, shared->x, (uint64_t)shared->tokens * k, "shared expert input", &sxr);
            if (st != FH_OK) return st;
            if (overlaps(sxr, syr) || overlaps(sxr, yr)) return fail(FH_ERR_RANGE, "expert output aliases an input");
        }
        if (overlaps(xr, syr) || overlaps(ir, syr) || overlaps(yr, syr))
            return fail(FH_ERR_RANGE, "shared expert output aliases another tensor");
    }
    GemvArgs a{};
    a.ggml_type = weight->ggml_type;
    a.w = weight->ptr;
    a.x = xr.begin;
    a.y = const_cast<uint8_t*>(yr.begin);
    a.n = (uint32_t)rows;
    a.k = (uint32_t)k;
    a.m = routes;
    a.x_dtype = x->dtype;
    a.y_dtype = y->dtype;
    a.metadata = reinterpret_cast<const float*>(ir.begin);
    a.meta_stride = 1;
    a.experts = (uint32_t)weight->experts;
    a.x_mode = kXDivide;
    a.x_div = x_div;
    a.x_rows = routes / x_div;
    if (shared != nullptr) {
        a.m = routes + shared->tokens;
        a.shared_w = shared->weight->ptr;
        a.shared_rows = shared->tokens;
        a.shared_x = sxr.begin;
        a.shared_y = const_cast<uint8_t*>(syr.begin);
    }
    const char* unused = "";
    st = run_gemv(device, a, &unused);
    if (st != FH_OK) return st;
    device->last_operation = weight->ggml_type == kQ4K     ? "h_mv_id_q4_k"
                             : weight->ggml_type == kQ5K   ? "h_mv_id_q5_k"
                             : weight->ggml_type == kQ6K   ? "h_mv_id_q6_k"
                             : weight->ggml_type == kQ8_0  ? "h_mv_id_q8_0"
                                                           : "h_mv_id_iq4_xs";
    FH_HIP(hipGetLastError());
    return FH_OK;
}

}  // namespace

fh_status fh_hybrid_project_id(fh_device* device, const fh_qmatrix* weight, const fh_view* x, const fh_view* ids,
                               uint32_t routes, uint32_t x_div, const fh_view* y) {
    return hybrid_project_id(device, weight, x, ids, routes, x_div, y, nullptr);
}

fh_status fh_hybrid_project_id_with_shared(fh_device* device, const fh_qmatrix* weight,
                                           const fh_qmatrix* shared_weight, const fh_view* x, const fh_view* ids,
                                           uint32_t routes, uint32_t x_div, uint32_t tokens, const fh_view* shared_x,
                                           const fh_view* y, const fh_view* shared_y) {
    if (shared_weight == nullptr || shared_y == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    SharedExpert shared;
    shared.weight = shared_weight;
    shared.tokens = tokens;
    shared.x = shared_x;
    shared.y = shared_y;
    return hybrid_project_id(device, weight, x, ids, routes, x_div, y, &shared);
}

fh_status fh_hybrid_moe_map(fh_device* device, const fh_view* ids, uint32_t experts, uint32_t routes,
                            const fh_view* offsets, const fh_view* sorted, const fh_view* position) {
    if (device == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (experts == 0 || experts > 1024 || routes == 0) return fail(FH_ERR_SHAPE, "route map needs 1..1024 experts and routes");
    for (const fh_view* v : {ids, offsets, sorted, position})
        if (v == nullptr || v->dtype != FH_F32) return fail(FH_ERR_DTYPE, "route map operands are f32 carriers of u32");
    Range ir, fr, sr, pr;
    fh_status st = resolve(device, ids, routes, "route ids", &ir, 4);
    if (st != FH_OK) return st;
    if ((st = resolve(device, offsets, (uint64_t)experts + 1, "expert offsets", &fr, 4)) != FH_OK) return st;
    if ((st = resolve(device, sorted, routes, "sorted routes", &sr, 4)) != FH_OK) return st;
    if ((st = resolve(device, position, routes, "route positions", &pr, 4)) != FH_OK) return st;
    if (overlaps(ir, fr) || overlaps(ir, sr) || overlaps(ir, pr) || overlaps(fr, sr) || overlaps(fr, pr) ||
        overlaps(sr, pr))
        return fail(FH_ERR_RANGE, "route map operands alias");
    auto words = [](const Range& r) { return reinterpret_cast<uint32_t*>(const_cast<uint8_t*>(r.begin)); };
    device->last_operation = launch_moe_map(device->stream, words(ir), experts, routes, words(fr), words(sr), words(pr));
    FH_HIP(hipGetLastError());
    return FH_OK;
}

fh_status fh_hybrid_moe_gather(fh_device* device, const fh_view* x, const fh_view* sorted, uint32_t hidden,
                               uint32_t used, uint32_t routes, const fh_view* out) {
    if (device == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (hidden == 0 || used == 0 || routes == 0 || routes % used != 0 || !fits_u32((uint64_t)routes * hidden))
        return fail(FH_ERR_SHAPE, "route gather needs [tokens, hidden] and tokens * used routes");
    if (sorted == nullptr || sorted->dtype != FH_F32 || x == nullptr || out == nullptr || out->dtype != x->dtype)
        return fail(FH_ERR_DTYPE, "route gather: sorted is an f32 carrier, output dtype is the input's");
    Range xr, sr, orr;
    fh_status st = resolve(device, x, (uint64_t)routes / used * hidden, "gather input", &xr);
    if (st != FH_OK) return st;
    if ((st = resolve(device, sorted, routes, "sorted routes", &sr, 4)) != FH_OK) return st;
    if ((st = resolve(device, out, (uint64_t)routes * hidden, "gather output", &orr)) != FH_OK) return st;
    if (overlaps(xr, orr) || overlaps(sr, orr)) return fail(FH_ERR_RANGE, "gather output aliases an input");
    device->last_operation = launch_moe_gather_sorted(
        device->stream, xr.begin, reinterpret_cast<const uint32_t*>(sr.begin), const_cast<uint8_t*>(orr.begin), routes,
        used, routes / used, hidden * (uint32_t)dtype_bytes(x->dtype));
    FH_HIP(hipGetLastError());
    return FH_OK;
}

namespace {

fh_status hybrid_project_mm_id(fh_device* device, const fh_qmatrix* weight, const fh_view* x,
                               const fh_view* offsets, uint32_t routes, const fh_view* y,
                               const SharedExpert* shared) {
    if (device == nullptr || weight == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (weight->device != device || routes == 0 || weight->experts > 1024 || offsets == nullptr ||
        offsets->dtype != FH_F32 || x == nullptr || y == nullptr)
        return fail(FH_ERR_SHAPE, "expert projection geometry");
    if (weight->padded()) {
        const fh_qmatrix stored = as_stored(weight);
        PaddedActivations pad(device, weight);
        PaddedRider pr;
        fh_view px{};
        pad.add(x, routes, "expert input", &px);
        if (shared != nullptr && shared->x == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
        fh_status pst = pad_rider(pad, weight, shared, 1, &pr);
        if (pst == FH_OK) pst = pad.run();
        if (pst == FH_OK) pst = pad.keep_apart(y, (uint64_t)routes * weight->rows, "expert output", "expert output aliases an input");
        if (pst == FH_OK && shared != nullptr)
            pst = pad.keep_apart(shared->y, (uint64_t)shared->tokens * weight->rows, "shared expert output",
                                 "shared expert output aliases another tensor");
        if (pst != FH_OK) return pst;
        return hybrid_project_mm_id(device, &stored, &px, offsets, routes, y, pr.get(shared));
    }
    const uint64_t rows = weight->rows, k = weight->cols;
    if (!fits_u32((uint64_t)routes * rows) || !fits_u32((uint64_t)routes * k))
        return fail(FH_ERR_SHAPE, "index does not fit in 32 bits");
    if ((rows * dtype_bytes(y->dtype)) % 4 != 0) return fail(FH_ERR_SHAPE, "expert output rows must be whole words");
    Range xr, fr, yr;
    fh_status st = resolve(device, x, (uint64_t)routes * k, "expert input", &xr);
    if (st != FH_OK) return st;
    if ((st = resolve(device, offsets, weight->experts + 1, "expert offsets", &fr, 4)) != FH_OK) return st;
    if ((st = resolve(device, y, (uint64_t)routes * rows, "expert output", &yr)) != FH_OK) return st;
    if (overlaps(xr, yr) || overlaps(fr, yr)) return fail(FH_ERR_RANGE, "expert output aliases an input");
    Range sxr{nullptr, 0}, syr{nullptr, 0};
    if (shared != nullptr) {
        const fh_qmatrix* sw = shared->weight;
        if (sw == nullptr || shared->x == nullptr || shared->y == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
        if (sw->device != device) {
            g_last_error = "weight belongs to another device";
            return FH_ERR_DEVICE_MISMATCH;
        }
        if (sw->experts != 1 || sw->rows != rows || sw->cols != k || sw->ggml_type != weight->ggml_type)
            return fail(FH_ERR_SHAPE, "the shared expert's matrix must have one expert's shape and format");
        if (shared->tokens == 0 || !fits_u32((uint64_t)shared->tokens * rows) || !fits_u32((uint64_t)shared->tokens * k))
            return fail(FH_ERR_SHAPE, "the shared expert runs once per token");
        if (shared->y->dtype != y->dtype || shared->x->dtype != x->dtype)
            return fail(FH_ERR_DTYPE, "the shared expert's tensors differ in dtype from the routed ones");
        if ((st = resolve(device, shared->x, (uint64_t)shared->tokens * k, "shared expert input", &sxr)) != FH_OK) return st;
        if ((st = resolve(device, shared->y, (uint64_t)shared->tokens * rows, "shared expert output", &syr)) != FH_OK)
            return st;
        if (overlaps(sxr, syr) || overlaps(sxr, yr) || overlaps(xr, syr) || overlaps(fr, syr) || overlaps(yr, syr))
            return fail(FH_ERR_RANGE, "shared expert output aliases another tensor");
        if (!expert_rows_fit_lds((uint32_t)k, routes, (uint32_t)weight->experts)) {
            // rows too wide for the kernel that carries the shared expert: the two run apart
            st = hybrid_project_mm_id(device, weight, x, offsets, routes, y, nullptr);
            if (st != FH_OK) return st;
            return project(device, shared->weight, shared->x, shared->tokens, shared->y, false, 5);
        }
    }
    // The tiles are f16 / bf16, as the reference's h_mm_id kernels make theirs.  f32 rows are rounded to f16
    // by the kernel that gathers them into LDS, or first where they are too wide for that one.
    const bool rounds_inside = x->dtype == FH_F32 && expert_rows_fit_lds((uint32_t)k, routes, (uint32_t)weight->experts);
    const void* tile_x = xr.begin;
    if (x->dtype == FH_F32 && !rounds_inside) {   // (a shared expert has left for its own call above)
        st = ensure_scratch(device, (size_t)routes * k * sizeof(uint16_t));
        if (st != FH_OK) return st;
        uint16_t* x16 = reinterpret_cast<uint16_t*>(scratch_data(device));
        launch_round_to_f16(device->stream, reinterpret_cast<const float*>(xr.begin), x16, (size_t)routes * k);
        tile_x = x16;
    }
    GemmArgs g{};
    g.ggml_type = weight->ggml_type;
    g.w = weight->ptr;
    g.x = tile_x;
    g.y = const_cast<uint8_t*>(yr.begin);
    g.n = (uint32_t)rows;
    g.k = (uint32_t)k;
    g.m = routes;
    g.x_dtype = x->dtype == FH_F32 ? FH_F16 : x->dtype;
    g.y_dtype = y->dtype;
    g.cu_count = device->props.multiProcessorCount;
    g.experts = (uint32_t)weight->experts;
    g.expert_offsets = reinterpret_cast<const uint32_t*>(fr.begin);
    g.expert_order = nullptr;   // rows are already expert-sorted
    g.x_rounds = rounds_inside;
    g.weight_ring = device->tuning.expert_weight_ring != 0;
    if (shared != nullptr) {
        g.shared_w = shared->weight->ptr;
        g.shared_rows = shared->tokens;
        g.shared_x = sxr.begin;
        g.shared_y = const_cast<uint8_t*>(syr.begin);
    }
    launch_gemm_skinny(device->stream, g);
    device->last_operation = weight->ggml_type == kQ4K     ? "h_mm_id_q4_k"
                             : weight->ggml_type == kQ5K   ? "h_mm_id_q5_k"
                             : weight->ggml_type == kQ6K   ? "h_mm_id_q6_k"
                             : weight->ggml_type == kQ8_0  ? "h_mm_id_q8_0"
                                                           : "h_mm_id_iq4_xs";
    FH_HIP(hipGetLastError());
    return FH_OK;
}

}  // namespace

fh_status fh_hybrid_project_mm_id(fh_device* device, const fh_qmatrix* weight, const fh_view* x,
                                  const fh_view* offsets, uint32_t routes, const fh_view* y) {
    return hybrid_project_mm_id(device, weight, x, offsets, routes, y, nullptr);
}

fh_status fh_hybrid_project_mm_id_with_shared(fh_device* device, const fh_qmatrix* weight,
                                              const fh_qmatrix* shared_weight, const fh_view* x,
                                              const fh_view* offsets, uint32_t routes, uint32_t tokens,
                                              const fh_view* shared_x, const fh_view* y, const fh_view* shared_y) {
    if (shared_weight == nullptr || shared_x == nullptr || shared_y == nullptr)
        return fail(FH_ERR_PARAMETER, "null argument");
    SharedExpert shared;
    shared.weight = shared_weight;
    shared.tokens = tokens;
    shared.x = shared_x;
    shared.y = shared_y;
    return hybrid_project_mm_id(device, weight, x, offsets, routes, y, &shared);
}

fh_status fh_hybrid_moe_combine(fh_device* device, const fh_view* down, const fh_view* weights,
                                const fh_view* position, const fh_view* shared, const fh_view* shared_gate,
                                uint32_t hidden, uint32_t used, uint32_t tokens, const fh_view* out) {
    if (device == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (hidden == 0 || used == 0 || tokens == 0 || !fits_u32((uint64_t)tokens * used * hidden))
        return fail(FH_ERR_SHAPE, "route combine needs [tokens * used, hidden]");
    for (const fh_view* v : {down, weights, shared, shared_gate, out})
        if (v == nullptr || v->dtype != FH_F32) return fail(FH_ERR_DTYPE, "the hybrid combine works on f32 rows");
    if (position != nullptr && position->dtype != FH_F32) return fail(FH_ERR_DTYPE, "positions are an f32 carrier of u32");
    const uint64_t routes = (uint64_t)tokens * used;
    Range dr, wr, pr{nullptr, 0}, sr, gr, orr;
    fh_status st = resolve(device, down, routes * hidden, "expert rows", &dr);
    if (st != FH_OK) return st;
    if ((st = resolve(device, weights, routes, "route weights", &wr, 4)) != FH_OK) return st;
    if (position != nullptr && (st = resolve(device, position, routes, "route positions", &pr, 4)) != FH_OK) return st;
    if ((st = resolve(device, shared, (uint64_t)tokens * hidden, "shared rows", &sr)) != FH_OK) return st;
    if ((st = resolve(device, shared_gate, tokens, "shared gate", &gr, 4)) != FH_OK) return st;
    if ((st = resolve(device, out, (uint64_t)tokens * hidden, "combine output", &orr)) != FH_OK) return st;
    if (overlaps(dr, orr) || overlaps(wr, orr) || overlaps(sr, orr) || overlaps(gr, orr) ||
        (position != nullptr && overlaps(pr, orr)))
        return fail(FH_ERR_RANGE, "combine output aliases an input");
    device->last_operation = launch_hybrid_combine(
        device->stream, reinterpret_cast<const float*>(dr.begin), reinterpret_cast<const float*>(wr.begin),
        reinterpret_cast<const uint32_t*>(pr.begin), reinterpret_cast<const float*>(sr.begin),
        reinterpret_cast<const float*>(gr.begin), reinterpret_cast<float*>(const_cast<uint8_t*>(orr.begin)), hidden, used,
        tokens, (uint32_t)routes);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

fh_status fh_expert_assign(fh_device* device, const fh_view* hidden, uint32_t tokens,
                           uint32_t width, const fh_view* metadata, uint32_t top_k,
                           const fh_view* out) {
    if (device == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (tokens == 0 || width == 0 || top_k == 0 || metadata == nullptr || metadata->dtype != FH_F32 ||
        !fits_u32((uint64_t)tokens * top_k) || !fits_u32((uint64_t)tokens * top_k * width))
        return fail(FH_ERR_SHAPE, "expert assignments require [S,H] and [S*top_k,3]");
    const uint32_t assignments = tokens * top_k;
    Range hr, mr, orr;
    fh_status st = resolve(device, hidden, (uint64_t)tokens * width, "assign input", &hr);
    if (st != FH_OK) return st;
    st = resolve(device, metadata, (uint64_t)assignments * 3, "assign metadata", &mr, 4);
    if (st != FH_OK) return st;
    st = resolve(device, out, (uint64_t)assignments * width, "assign output", &orr);
    if (st != FH_OK) return st;
    if (out->dtype != hidden->dtype) return fail(FH_ERR_DTYPE, "assign output dtype differs from input");
    if (overlaps(hr, orr) || overlaps(mr, orr)) return fail(FH_ERR_RANGE, "assign output aliases an input");
    device->last_operation = launch_expert_assign(
        device->stream, hr.begin, reinterpret_cast<const float*>(mr.begin),
        const_cast<uint8_t*>(orr.begin), assignments, width * (uint32_t)dtype_bytes(hidden->dtype), tokens);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

namespace {

// Whether one per-assignment launch takes this many entries.  Such a launch is not cut into runs while a shared
// expert rides in it, so it ends with the grid's z extent and, where a long row's K is cut into segments, with
// the counter words (one per row tile and entry: 4096 x 7168 matrices reach that at 128 entries).
bool rider_fits(uint32_t n, uint32_t k, uint64_t entries) {
    const GemvPlan plan = gemv_plan(n, k, 1, 0);
    return entries <= 65535u && (plan.segments <= 1 || plan.tiles * entries <= fh_device::kCounterWords);
}

// Whether streaming every hit expert once for all of its rows beats streaming it once per row.  The
// per-assignment launch reads an expert's matrix for each of its assignments at the rate of its decode (rows
// whose super-blocks leave more than a third of the kernel's block slots idle, as five on eight do, a fifth
// below it); the grouped one waits for the workgroup that streams one share of one expert, behind a grouping
// and a staging launch (9 and 15.5 us before either streams).  One projection, f16, us, per assignment against grouped: 64 experts of 2048 x 1280, 64 /
// 96 / 128 assignments Q4_K 28 / 36 / 44 against 32, IQ4_XS 37 / 50 / 62 against 38; 128 of 2048 x 768, 128 / 192 /
// 256 Q4_K 25 / 32 / 40 against 35, IQ4_XS 35 / 47 / 60 against 44; 256 of 1024 x 2048, 256 / 384 Q6_K 81 / 124
// against 117.  From five assignments per expert on they are grouped.
bool grouping_pays(const fh_qmatrix& weight, uint32_t assignments, int cu_count) {
    if (assignments >= 5 * weight.experts) return true;
    struct Rates { double each, share; };   // bytes per us: of the chip, and of a compute unit that multiplies groups
    const Rates rates = weight.ggml_type == kQ4K    ? Rates{6.4e6, 21.0e3}
                        : weight.ggml_type == kQ5K  ? Rates{5.9e6, 17.0e3}
                        : weight.ggml_type == kQ6K  ? Rates{5.9e6, 16.5e3}
                        : weight.ggml_type == kQ8_0 ? Rates{7.8e6, 25.0e3}
                                                    : Rates{4.4e6, 14.5e3};
    const uint32_t nb = (uint32_t)(weight.stored_cols / 256);
    const GemvPlan plan = gemv_plan((uint32_t)weight.rows, nb * 256, 1, 0);
    const bool idles = plan.segments * (uint32_t)(plan.bs * plan.it) * 2 >= nb * 3;
    const double bytes = (double)weight.rows * nb * block_bytes(weight.ggml_type);
    const double shares = std::max(1.0, (double)cu_count / (double)weight.experts);
    return 9.0 + assignments * bytes / rates.each * (idles ? 1.2 : 1.0) > 15.5 + bytes / (shares * rates.share);
}

fh_status expert_project(fh_device* device, const fh_qmatrix* weight, const fh_view* x, uint32_t x_rows,
                         uint32_t form, uint32_t assignments, const fh_view* metadata, const fh_view* y,
                         const SharedExpert* shared = nullptr, const RouteTokenArgs* route = nullptr,
                         bool grouped_before = false) {
    // grouped_before: the grouped form finds offsets and order of these very records (all ids valid)
    // at the head of the scratch, left there by the call before; the scratch must not grow in between
    if (device == nullptr || weight == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (form > FH_INPUT_SILU_MUL) return fail(FH_ERR_PARAMETER, "unknown input form %u", form);
    if (shared != nullptr && form == FH_INPUT_ROWS)
        return fail(FH_ERR_PARAMETER, "a shared expert needs the gathered or the SiLU input form");
    if (form == FH_INPUT_GATHER && x_rows == 0) return fail(FH_ERR_SHAPE, "gathered expert projection needs tokens");
    if (weight->device != device || assignments == 0 || metadata == nullptr ||
        metadata->dtype != FH_F32 || metadata->buffer == nullptr ||
        metadata->buffer->device != device || x == nullptr || x->buffer == nullptr ||
        x->buffer->device != device)
        return fail(FH_ERR_SHAPE, "quantized expert projection geometry mismatch");
    if (weight->padded()) {
        if (route != nullptr || grouped_before)
            return fail(FH_ERR_DISPATCH, "a matrix whose rows are stored padded takes the separate launches");
        if (shared != nullptr && (form == FH_INPUT_SILU_MUL) != (shared->x != nullptr))
            return fail(FH_ERR_PARAMETER, "the shared expert takes its own input in the SiLU form only");
        const fh_qmatrix stored = as_stored(weight);
        PaddedActivations pad(device, weight);
        PaddedRider pr;
        fh_view px{};
        const uint32_t parts = form == FH_INPUT_SILU_MUL ? 2 : 1;
        pad.add(x, form == FH_INPUT_GATHER ? (uint64_t)x_rows : (uint64_t)assignments * parts, "expert input", &px);
        fh_status pst = pad_rider(pad, weight, shared, parts, &pr);
        if (pst == FH_OK) pst = pad.run();
        if (pst == FH_OK)
            pst = pad.keep_apart(y, (uint64_t)assignments * weight->rows, "expert output", "expert output aliases an input");
        if (pst == FH_OK && shared != nullptr)
            pst = pad.keep_apart(shared->y, (uint64_t)shared->tokens * weight->rows, "shared expert output",
                                 "shared expert output aliases another tensor");
        if (pst != FH_OK) return pst;
        return expert_project(device, &stored, &px, x_rows, form, assignments, metadata, y, pr.get(shared));
    }
    const uint64_t rows = weight->rows, k = weight->cols;
    // elements the input view must hold: [A,K], [tokens,K] or [A,2K]
    const uint64_t x_elements = form == FH_INPUT_GATHER ? (uint64_t)x_rows * k
                                : (uint64_t)assignments * k * (form == FH_INPUT_SILU_MUL ? 2 : 1);
    if (!fits_u32((uint64_t)assignments * rows) || !fits_u32(x_elements))
        return fail(FH_ERR_SHAPE, "index does not fit in 32 bits");
    Range xr, mr, yr;
    fh_status st = resolve(device, x, x_elements, "expert input", &xr);
    if (st != FH_OK) return st;
    st = resolve(device, metadata, (uint64_t)assignments * 3, "expert metadata", &mr, 4);
    if (st != FH_OK) return st;
    st = resolve(device, y, (uint64_t)assignments * rows, "expert output", &yr);
    if (st != FH_OK) return st;
    if (overlaps(xr, yr) || overlaps(mr, yr)) return fail(FH_ERR_RANGE, "expert output aliases an input");
    Range sxr{nullptr, 0}, syr{nullptr, 0};
    if (shared != nullptr) {
        const fh_qmatrix* sw = shared->weight;
        if (sw == nullptr || shared->y == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
        if (sw->device != device) {
            g_last_error = "weight belongs to another device";
            return FH_ERR_DEVICE_MISMATCH;
        }
        if (sw->experts != 1 || sw->rows != rows || sw->cols != k || sw->ggml_type != weight->ggml_type)
            return fail(FH_ERR_SHAPE, "the shared expert's matrix must have one expert's shape and format");
        if (shared->tokens == 0 || (form == FH_INPUT_GATHER && shared->tokens != x_rows) ||
            !fits_u32((uint64_t)assignments + shared->tokens) || !fits_u32((uint64_t)shared->tokens * rows))
            return fail(FH_ERR_SHAPE, "the shared expert runs once per token");
        if ((form == FH_INPUT_SILU_MUL) != (shared->x != nullptr))
            return fail(FH_ERR_PARAMETER, "the shared expert takes its own input in the SiLU form only");
        if (shared->y->dtype != y->dtype || (shared->x != nullptr && shared->x->dtype != x->dtype))
            return fail(FH_ERR_DTYPE, "the shared expert's tensors differ in dtype from the routed ones");
        st = resolve(device, shared->y, (uint64_t)shared->tokens * rows, "shared expert output", &syr);
        if (st != FH_OK) return st;
        if (shared->x != nullptr) {
            st = resolve(device, shared->x, (uint64_t)shared->tokens * k * 2, "shared expert input", &sxr);
            if (st != FH_OK) return st;
            if (overlaps(sxr, syr) || overlaps(sxr, yr)) return fail(FH_ERR_RANGE, "expert output aliases an input");
        }
        if (overlaps(xr, syr) || overlaps(mr, syr) || overlaps(yr, syr))
            return fail(FH_ERR_RANGE, "shared expert output aliases another tensor");
    }
    const int64_t grouped_min = device->tuning.expert_grouped_min_assignments;
    // f32 rows join the grouped form when the caller has opted f32 activations into the f16
    // tiles (gemm_f32_min_rows, the hybrid engine's prompt path project_mm_id_in,
    // src/hybrid/engine.rs:3164): they are rounded to f16 into the scratch first
    const int64_t f32_rows = device->tuning.gemm_f32_min_rows;
    const bool f32_grouped = form == FH_INPUT_ROWS && x->dtype == FH_F32 && f32_rows > 0 &&
                             assignments >= (uint64_t)f32_rows && ((uintptr_t)xr.begin & 15u) == 0;
    const bool grouped = (x->dtype != FH_F32 || f32_grouped) && grouped_min > 0 &&
                         assignments >= (uint64_t)grouped_min &&
                         (f32_grouped || grouping_pays(*weight, assignments, device->props.multiProcessorCount)) &&
                         weight->experts <= 1024 &&
                         (rows * dtype_bytes(y->dtype)) % 4 == 0;
    if (grouped && route != nullptr) return fail(FH_ERR_DISPATCH, "only the per-assignment launch routes its token");
    if (shared != nullptr &&
        (grouped ? !expert_rows_fit_lds((uint32_t)k, assignments, (uint32_t)weight->experts)
                 : !rider_fits((uint32_t)rows, (uint32_t)k, (uint64_t)assignments + shared->tokens))) {
        // A shared expert rides in the grouped form only in the kernel that keeps rows in LDS, and in the
        // per-assignment form only where the launch need not be cut into runs: otherwise the two run apart, as
        // the separate calls would.
        st = expert_project(device, weight, x, x_rows, form, assignments, metadata, y, nullptr, route);
        if (st != FH_OK) return st;
        if (form == FH_INPUT_GATHER) return project(device, shared->weight, x, shared->tokens, shared->y, false);
        if (shared->tokens < (uint64_t)device->tuning.gemm_min_rows || x->dtype == FH_F32 ||
            ((uintptr_t)sxr.begin & 15u) != 0)
            return project(device, shared->weight, shared->x, shared->tokens, shared->y, true);
        GemmArgs g = gemm_args(device, weight->ggml_type, rows, k, shared->tokens, x->dtype, y->dtype);
        if (!gemm_takes_rows(g)) gemm_takes_decoded(g);
        st = prepare_gemm(device, g, (size_t)shared->tokens * k * sizeof(uint16_t));
        if (st != FH_OK) return st;
        launch_expert_silu_mul(device->stream, sxr.begin, scratch_data(device), shared->tokens, (uint32_t)k, x->dtype,
                               x->dtype);
        g.w = shared->weight->ptr;
        g.x = scratch_data(device);
        g.y = const_cast<uint8_t*>(syr.begin);
        device->last_operation = run_gemm(device, g);
        FH_HIP(hipGetLastError());
        return FH_OK;
    }
    if (grouped) {
        // grouped form: every expert's weights are streamed once for all of its assignments.
        // The kernel that keeps an expert's rows in LDS gathers them from the token rows
        // itself; where they do not fit, and for the SiLU form, the rows are written out
        // first, as the separate expert_assign / expert_silu_mul launches would.
        const bool gathers = form == FH_INPUT_GATHER &&
                             expert_rows_fit_lds((uint32_t)k, assignments, (uint32_t)weight->experts);
        const bool staged = f32_grouped || (form != FH_INPUT_ROWS && !gathers);
        const size_t words = ((size_t)weight->experts + 1 + assignments + 3) & ~(size_t)3;
        // the SiLU form stages the shared expert's rows behind the routed ones
        const size_t staged_rows = (size_t)assignments + (shared != nullptr && form == FH_INPUT_SILU_MUL ? shared->tokens : 0);
        const size_t staged_bytes = staged ? staged_rows * k * sizeof(uint16_t) : 0;
        st = ensure_scratch(device, words * sizeof(uint32_t) + staged_bytes);
        if (st != FH_OK) return st;
        uint32_t* offsets = reinterpret_cast<uint32_t*>(scratch_data(device));
        uint32_t* order = offsets + weight->experts + 1;
        const void* tile_x = xr.begin;
        uint8_t* shared_rows_x = nullptr;  // the shared expert's own rows, when it does not read the token rows
        if (staged) {
            uint8_t* rows_x = scratch_data(device) + words * sizeof(uint32_t);
            if (f32_grouped) {
                launch_round_to_f16(device->stream, reinterpret_cast<const float*>(xr.begin),
                                    reinterpret_cast<uint16_t*>(rows_x), (size_t)assignments * k);
            } else if (form == FH_INPUT_GATHER) {
                launch_expert_assign(device->stream, xr.begin, reinterpret_cast<const float*>(mr.begin), rows_x,
                                     assignments, (uint32_t)(k * sizeof(uint16_t)), x_rows);
            } else if (shared != nullptr) {
                shared_rows_x = rows_x + (size_t)assignments * k * sizeof(uint16_t);
                launch_expert_silu_mul_pair(device->stream, xr.begin, sxr.begin, rows_x, assignments, shared->tokens,
                                            (uint32_t)k, x->dtype);
            } else {
                launch_expert_silu_mul(device->stream, xr.begin, rows_x, assignments, (uint32_t)k, x->dtype,
                                       x->dtype);
            }
            tile_x = rows_x;
        }
        if (!grouped_before)
            launch_expert_group(device->stream, reinterpret_cast<const float*>(mr.begin), assignments,
                                (uint32_t)weight->experts, offsets, order, const_cast<uint8_t*>(yr.begin),
                                (uint32_t)(rows * dtype_bytes(y->dtype)));
        GemmArgs g{};
        g.ggml_type = weight->ggml_type;
        g.w = weight->ptr;
        g.x = tile_x;
        g.y = const_cast<uint8_t*>(yr.begin);
        g.n = (uint32_t)rows;
        g.k = (uint32_t)k;
        g.m = assignments;
        g.x_dtype = f32_grouped ? FH_F16 : x->dtype;
        g.y_dtype = y->dtype;
        g.cu_count = device->props.multiProcessorCount;
        g.experts = (uint32_t)weight->experts;
        g.expert_offsets = offsets;
        g.expert_order = order;
        g.gather_metadata = gathers ? reinterpret_cast<const float*>(mr.begin) : nullptr;
        g.x_rows = x_rows;
        g.weight_ring = device->tuning.expert_weight_ring != 0;
        if (shared != nullptr) {
            g.shared_w = shared->weight->ptr;
            g.shared_rows = shared->tokens;
            // gathered form: the token rows themselves, in place or as staged for the routed rows' gather
            g.shared_x = form == FH_INPUT_GATHER ? xr.begin : shared_rows_x;
            g.shared_y = const_cast<uint8_t*>(syr.begin);
        }
        device->last_operation = launch_gemm_skinny(device->stream, g);
        FH_HIP(hipGetLastError());
        return FH_OK;
    }
    GemvArgs a{};
    a.ggml_type = weight->ggml_type;
    a.w = weight->ptr;
    a.x = xr.begin;
    a.y = const_cast<uint8_t*>(yr.begin);
    a.n = (uint32_t)rows;
    a.k = (uint32_t)k;
    a.m = assignments;
    a.x_dtype = x->dtype;
    a.y_dtype = y->dtype;
    a.metadata = reinterpret_cast<const float*>(mr.begin);
    a.experts = (uint32_t)weight->experts;
    a.ksplit = 0;
    a.x_mode = form;
    a.x_rows = form == FH_INPUT_GATHER ? x_rows : assignments;
    a.route = route;
    if (shared != nullptr) {
        a.m = assignments + shared->tokens;
        a.shared_w = shared->weight->ptr;
        a.shared_rows = shared->tokens;
        a.shared_x = sxr.begin;
        a.shared_y = const_cast<uint8_t*>(syr.begin);
    }
    const char* name = "";
    st = run_gemv(device, a, &name);
    if (st != FH_OK) return st;
    device->last_operation = name;
    FH_HIP(hipGetLastError());
    return FH_OK;
}

}  // namespace

fh_status fh_expert_project_with_shared(fh_device* device, const fh_qmatrix* weight,
                                        const fh_qmatrix* shared_weight, const fh_view* x, uint32_t tokens,
                                        uint32_t input_form, uint32_t assignments, const fh_view* metadata,
                                        const fh_view* shared_x, const fh_view* y, const fh_view* shared_y) {
    SharedExpert shared;
    shared.weight = shared_weight;
    shared.tokens = tokens;
    shared.x = shared_x;
    shared.y = shared_y;
    if (shared_weight == nullptr || shared_y == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    return expert_project(device, weight, x, tokens, input_form, assignments, metadata, y, &shared);
}

fh_status fh_expert_project_quantized(fh_device* device, const fh_qmatrix* weight,
                                      const fh_view* x, uint32_t assignments,
                                      const fh_view* metadata, const fh_view* y) {
    return expert_project(device, weight, x, assignments, FH_INPUT_ROWS, assignments, metadata, y);
}

fh_status fh_expert_project_fused(fh_device* device, const fh_qmatrix* weight, const fh_view* x,
                                  uint32_t x_rows, uint32_t input_form, uint32_t assignments,
                                  const fh_view* metadata, const fh_view* y) {
    return expert_project(device, weight, x, x_rows, input_form, assignments, metadata, y);
}

fh_status fh_expert_silu_mul(fh_device* device, const fh_view* in, uint32_t assignments,
                             uint32_t intermediate, const fh_view* out) {
    if (device == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (assignments == 0 || intermediate == 0 || !fits_u32((uint64_t)assignments * intermediate * 2))
        return fail(FH_ERR_SHAPE, "packed expert activation geometry mismatch");
    Range ir, orr;
    fh_status st = resolve(device, in, (uint64_t)assignments * intermediate * 2, "silu_mul input", &ir, 4);
    if (st != FH_OK) return st;
    st = resolve(device, out, (uint64_t)assignments * intermediate, "silu_mul output", &orr, 4);
    if (st != FH_OK) return st;
    if (overlaps(ir, orr)) return fail(FH_ERR_RANGE, "silu_mul output aliases its input");
    device->last_operation = launch_expert_silu_mul(device->stream, ir.begin,
                                                    const_cast<uint8_t*>(orr.begin), assignments,
                                                    intermediate, in->dtype, out->dtype);
    FH_HIP(hipGetLastError());
    return FH_OK;
}

namespace {

fh_status combine(fh_device* device, const fh_view* in, const fh_view* metadata, uint32_t tokens, uint32_t hidden,
                  uint32_t top_k, const fh_view* shared, const fh_view* shared_gate, const fh_view* out) {
    if (device == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    if (top_k == 0 || hidden == 0 || tokens == 0 || metadata == nullptr || metadata->dtype != FH_F32 ||
        !fits_u32((uint64_t)tokens * top_k * hidden))
        return fail(FH_ERR_SHAPE, "expert combine geometry mismatch");
    Range ir, mr, orr, sr{nullptr, 0}, gr{nullptr, 0};
    fh_status st = resolve(device, in, (uint64_t)tokens * top_k * hidden, "combine input", &ir, 4);
    if (st != FH_OK) return st;
    st = resolve(device, metadata, (uint64_t)tokens * top_k * 3, "combine metadata", &mr, 4);
    if (st != FH_OK) return st;
    st = resolve(device, out, (uint64_t)tokens * hidden, "combine output", &orr, 4);
    if (st != FH_OK) return st;
    if (overlaps(ir, orr) || overlaps(mr, orr)) return fail(FH_ERR_RANGE, "combine output aliases an input");
    if (shared != nullptr) {
        if (shared->dtype != in->dtype) return fail(FH_ERR_DTYPE, "the shared expert's output has the dtype of the routed rows");
        st = resolve(device, shared, (uint64_t)tokens * hidden, "shared expert output", &sr, 4);
        if (st != FH_OK) return st;
        if (overlaps(sr, orr)) return fail(FH_ERR_RANGE, "combine output aliases an input");
        if (shared_gate != nullptr) {
            if (shared_gate->dtype != FH_F32) return fail(FH_ERR_DTYPE, "the shared-expert gate is f32");
            st = resolve(device, shared_gate, tokens, "shared-expert gate", &gr, 4);
            if (st != FH_OK) return st;
        }
    }
    device->last_operation = launch_expert_combine(
        device->stream, ir.begin, reinterpret_cast<const float*>(mr.begin),
        const_cast<uint8_t*>(orr.begin), tokens, hidden, top_k, in->dtype, out->dtype, sr.begin,
        reinterpret_cast<const float*>(gr.begin));
    FH_HIP(hipGetLastError());
    return FH_OK;
}

}  // namespace

fh_status fh_expert_combine(fh_device* device, const fh_view* in, const fh_view* metadata,
                            uint32_t tokens, uint32_t hidden, uint32_t top_k, const fh_view* out) {
    return combine(device, in, metadata, tokens, hidden, top_k, nullptr, nullptr, out);
}

fh_status fh_expert_combine_shared(fh_device* device, const fh_view* in, const fh_view* metadata,
                                   uint32_t tokens, uint32_t hidden, uint32_t top_k, const fh_view* shared,
                                   const fh_view* shared_gate, const fh_view* out) {
    if (shared == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    return combine(device, in, metadata, tokens, hidden, top_k, shared, shared_gate, out);
}

// ---- the routed FFN in one call ------------------------------------------------------------

namespace {

fh_status ensure_workspace(fh_device* d, size_t bytes) {
    return ensure_block(d, d->workspace, bytes, "the routed FFN's workspace");
}

}  // namespace

fh_status fh_moe_ffn(fh_device* device, const fh_view* hidden, const fh_view* router_logits, uint32_t tokens,
                     const fh_view* selection_bias, const fh_routing_policy* policy,
                     const fh_qmatrix* input_experts, const fh_qmatrix* output_experts,
                     const fh_qmatrix* shared_input, const fh_qmatrix* shared_output,
                     const fh_view* shared_gate, const fh_view* out) {
    if (device == nullptr || hidden == nullptr || router_logits == nullptr || policy == nullptr ||
        input_experts == nullptr || output_experts == nullptr || out == nullptr)
        return fail(FH_ERR_PARAMETER, "null argument");
    // SparseMoe::new's geometry checks (src/nn/moe.rs:137-181)
    const uint64_t e = input_experts->experts, two_i = input_experts->rows, h = input_experts->cols;
    if (tokens == 0 || two_i == 0 || two_i % 2 != 0 || output_experts->experts != e || output_experts->rows != h ||
        output_experts->cols * 2 != two_i || policy->experts != e || policy->top_k == 0 || policy->top_k > e ||
        input_experts->device != device || output_experts->device != device)
        return fail(FH_ERR_SHAPE, "invalid sparse expert weight geometry");
    const bool shared = shared_input != nullptr;
    if ((shared_input == nullptr) != (shared_output == nullptr) ||
        (shared && (shared_input->cols != h || shared_output->rows != h || shared_input->rows == 0 ||
                    shared_input->rows != 2 * shared_output->cols || shared_input->experts != 1 ||
                    shared_output->experts != 1 || shared_input->device != device || shared_output->device != device)))
        return fail(FH_ERR_SHAPE, "invalid shared expert weight geometry");
    if (!shared && shared_gate != nullptr) return fail(FH_ERR_PARAMETER, "a shared gate without a shared expert");
    if (out->dtype != hidden->dtype) return fail(FH_ERR_DTYPE, "the routed FFN writes the activation dtype");
    const uint32_t k = policy->top_k, dt = hidden->dtype;
    const size_t es = dtype_bytes(dt), inter = (size_t)two_i / 2, si = shared ? (size_t)shared_output->cols : 0;
    // matrices whose rows are stored padded take the separate launches, each padding its own activations
    const bool stored_padded = input_experts->padded() || output_experts->padded() ||
                               (shared && (shared_input->padded() || shared_output->padded()));
    const bool rides = shared && shared_input->rows == two_i && shared_input->ggml_type == input_experts->ggml_type &&
                       shared_output->ggml_type == output_experts->ggml_type;

    // tokens are taken in chunks whose routing temporaries stay under the limit (src/nn/moe.rs:232-256)
    const size_t per_assignment = (2 * (size_t)h + 3 * inter) * es + 3 * sizeof(float);
    const size_t per_token = per_assignment * k + ((size_t)e + (size_t)h) * es;
    const size_t limit = (size_t)device->tuning.moe_routing_temporary_limit;
    const uint32_t chunk = (uint32_t)std::min<size_t>(tokens, std::max<size_t>(1, limit / per_token));

    // workspace layout for one chunk
    const size_t a_max = (size_t)chunk * k;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        const size_t here = at;
        at += align256(bytes);
        return here;
    };
    const size_t meta_at = take(a_max * 3 * sizeof(float));
    const size_t assigned_at = take(a_max * h * es);
    const size_t projected_at = take(a_max * two_i * es);
    const size_t activated_at = take(a_max * inter * es);
    const size_t expert_out_at = take(a_max * h * es);
    const size_t sproj_at = take(shared ? (size_t)chunk * 2 * si * es : 0);
    const size_t sact_at = take(shared ? (size_t)chunk * si * es : 0);
    const size_t sout_at = take(shared ? (size_t)chunk * h * es : 0);
    fh_status st = ensure_workspace(device, at);
    if (st != FH_OK) return st;
    fh_buffer* ws = device->workspace;
    auto view = [&](size_t offset, uint32_t dtype) { return fh_view{ws, offset, dtype}; };

    for (uint32_t start = 0; start < tokens; start += chunk) {
        const uint32_t count = std::min(chunk, tokens - start);
        const uint32_t a = count * k;
        const fh_view x = {hidden->buffer, hidden->offset + (size_t)start * h * es, dt};
        const fh_view logits = {router_logits->buffer,
                                router_logits->offset + (size_t)start * e * dtype_bytes(router_logits->dtype),
                                router_logits->dtype};
        const fh_view y = {out->buffer, out->offset + (size_t)start * h * es, dt};
        fh_view gate{};
        if (shared_gate) gate = {shared_gate->buffer, shared_gate->offset + (size_t)start * sizeof(float), shared_gate->dtype};
        const fh_view meta = view(meta_at, FH_F32), assigned = view(assigned_at, dt), projected = view(projected_at, dt),
                      activated = view(activated_at, dt), expert_out = view(expert_out_at, dt),
                      sproj = view(sproj_at, dt), sact = view(sact_at, dt), sout = view(sout_at, dt);
        // the copy and the activation ride inside the projections: per assignment in decode, in
        // the grouped kernel's gather of an expert's rows beyond it (f32 rows have no grouped form)
        const bool fused = a <= 31 || dt != FH_F32;
        // One token: the down projection of its entries and the weighted sum over them are one
        // launch (the bits of the two; 17.1 against 18.4 us for the 256-expert top-8 FFN with a
        // shared expert).  From two tokens on the two launches are the faster way (22.1 against
        // 23.2 us): the projection's launch stages an entry's activations once for 32 rows, this one
        // once for 8.
        const bool folded = count == 1 && a <= 31 && (!shared || rides) && !stored_padded &&
                            device->tuning.moe_fold_combine != 0 &&
                            (!shared_gate || shared_gate->dtype == FH_F32) &&
                            expert_down_combine_fits(output_experts->ggml_type, (uint32_t)h, (uint32_t)inter, k, shared);
        // ... and so does the routing: every workgroup of the gate|up launch routes the token
        // itself before it asks for its expert's rows, which takes a launch and the wait for its
        // records out of the chain
        const int64_t grouped_from = device->tuning.expert_grouped_min_assignments;
        const bool routes_inside = folded && device->tuning.moe_fold_route != 0 &&
                                   (grouped_from <= 0 || a < (uint64_t)grouped_from) &&   // the per-assignment launch
                                   gemv_routes((uint32_t)two_i, (uint32_t)h, (uint32_t)e, k);
        RouteTokenArgs inside{};
        st = route(device, &logits, count, selection_bias, policy, &meta, false, nullptr, nullptr, 0, nullptr, nullptr,
                   nullptr, routes_inside ? &inside : nullptr);
        if (st != FH_OK) return st;
        if (folded) {
            SharedExpert rider;
            rider.weight = shared_input;
            rider.tokens = count;
            rider.x = nullptr;
            rider.y = &sproj;
            st = expert_project(device, input_experts, &x, count, FH_INPUT_GATHER, a, &meta, &projected,
                                shared ? &rider : nullptr, routes_inside ? &inside : nullptr);
            if (st != FH_OK) return st;
            Range yr, gr{nullptr, 0};
            st = resolve(device, &y, (uint64_t)count * h, "routed FFN output", &yr);
            if (st != FH_OK) return st;
            if (shared_gate) {
                st = resolve(device, &gate, count, "shared-expert gate", &gr, 4);
                if (st != FH_OK) return st;
            }
            ExpertDownCombineArgs d{};
            d.ggml_type = output_experts->ggml_type;
            d.w = output_experts->ptr;
            d.w_shared = shared ? shared_output->ptr : nullptr;
            d.x = static_cast<const uint8_t*>(ws->ptr) + projected_at;
            d.x_shared = shared ? static_cast<const uint8_t*>(ws->ptr) + sproj_at : nullptr;
            d.metadata = reinterpret_cast<const float*>(static_cast<const uint8_t*>(ws->ptr) + meta_at);
            d.shared_gate = reinterpret_cast<const float*>(gr.begin);
            d.y = const_cast<uint8_t*>(yr.begin);
            d.n = (uint32_t)h;
            d.k = (uint32_t)inter;
            d.tokens = count;
            d.top_k = k;
            d.experts = (uint32_t)e;
            d.dtype = dt;
            device->last_operation = launch_expert_down_combine(device->stream, d);
            FH_HIP(hipGetLastError());
            continue;
        }
        // Both projections of a chunk group the same records by expert: the second finds the first's
        // offsets and order at the head of the scratch (the router's ids are all valid, and the scratch
        // is brought to the larger call's size before the first, so it does not move in between).
        const int64_t group_from = device->tuning.expert_grouped_min_assignments;
        // (With a shared expert whose rows do not fit LDS a projection runs the shared matrix as a dense call of its
        // own after the grouping, and that call may put partial sums where the lists lie: both then group for themselves.)
        const bool shared_stays_inside = !shared || (rides && expert_rows_fit_lds((uint32_t)h, a, (uint32_t)e) &&
                                                     expert_rows_fit_lds((uint32_t)inter, a, (uint32_t)e));
        const int cus = device->props.multiProcessorCount;
        const bool regroup_once = fused && dt != FH_F32 && group_from > 0 && a >= (uint64_t)group_from && e <= 1024 &&
                                  shared_stays_inside && !stored_padded && grouping_pays(*input_experts, a, cus) &&
                                  grouping_pays(*output_experts, a, cus);
        if (regroup_once) {
            const size_t words = ((size_t)e + 1 + a + 3) & ~(size_t)3;
            const size_t widest = std::max<size_t>(h, inter);
            st = ensure_scratch(device, words * sizeof(uint32_t) + ((size_t)a + count) * widest * sizeof(uint16_t));
            if (st != FH_OK) return st;
        }
        if (shared && rides && fused) {
            SharedExpert in_rider, out_rider;
            in_rider.weight = shared_input;
            in_rider.tokens = count;
            in_rider.y = &sproj;
            out_rider.weight = shared_output;
            out_rider.tokens = count;
            out_rider.x = &sproj;
            out_rider.y = &sout;
            st = expert_project(device, input_experts, &x, count, FH_INPUT_GATHER, a, &meta, &projected, &in_rider);
            if (st != FH_OK) return st;
            st = expert_project(device, output_experts, &projected, count, FH_INPUT_SILU_MUL, a, &meta, &expert_out,
                                &out_rider, nullptr, regroup_once);
            if (st != FH_OK) return st;
        } else {
            if (fused) {
                st = expert_project(device, input_experts, &x, count, FH_INPUT_GATHER, a, &meta, &projected);
                if (st != FH_OK) return st;
                st = expert_project(device, output_experts, &projected, a, FH_INPUT_SILU_MUL, a, &meta, &expert_out,
                                    nullptr, nullptr, regroup_once);
                if (st != FH_OK) return st;
            } else {
                st = fh_expert_assign(device, &x, count, (uint32_t)h, &meta, k, &assigned);
                if (st != FH_OK) return st;
                st = fh_expert_project_quantized(device, input_experts, &assigned, a, &meta, &projected);
                if (st != FH_OK) return st;
                st = fh_expert_silu_mul(device, &projected, a, (uint32_t)inter, &activated);
                if (st != FH_OK) return st;
                st = fh_expert_project_quantized(device, output_experts, &activated, a, &meta, &expert_out);
                if (st != FH_OK) return st;
            }
            if (shared) {
                st = fh_project_quantized(device, shared_input, &x, count, &sproj);
                if (st != FH_OK) return st;
                if (count <= 31) {
                    st = fh_project_silu_mul_quantized(device, shared_output, &sproj, count, &sout);
                } else {
                    st = fh_expert_silu_mul(device, &sproj, count, (uint32_t)si, &sact);
                    if (st != FH_OK) return st;
                    st = fh_project_quantized(device, shared_output, &sact, count, &sout);
                }
                if (st != FH_OK) return st;
            }
        }
        st = shared ? fh_expert_combine_shared(device, &expert_out, &meta, count, (uint32_t)h, k, &sout,
                                               shared_gate ? &gate : nullptr, &y)
                    : fh_expert_combine(device, &expert_out, &meta, count, (uint32_t)h, k, &y);
        if (st != FH_OK) return st;
    }
    return FH_OK;
}

// ---- batched execution ---------------------------------------------------------------

fh_status fh_execution_begin(fh_device* device) {
    if (device == nullptr) return fail(FH_ERR_PARAMETER, "null device");
    if (device->capturing) return fail(FH_ERR_DISPATCH, "nested executions are not supported");
    std::lock_guard<std::mutex> alone(device->freed.settling);   // no thread is waiting for the GPU to empty the pool
    std::lock_guard<std::mutex> hold(device->freed.lock);
    FH_HIP(hipStreamBeginCapture(device->stream, hipStreamCaptureModeThreadLocal));
    device->capturing = true;
    return FH_OK;
}

fh_status fh_execution_end(fh_device* device, fh_graph** out) {
    if (device == nullptr || out == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    *out = nullptr;
    if (!device->capturing) return fail(FH_ERR_DISPATCH, "no execution is being recorded");
    device->capturing = false;
    hipGraph_t graph = nullptr;
    const hipError_t ended = hipStreamEndCapture(device->stream, &graph);
    drain_deferred(device);
    if (ended != hipSuccess) return hip_fail(ended, "hipStreamEndCapture");
    hipGraphExec_t exec = nullptr;
    hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    if (e != hipSuccess) {
        (void)hipGraphDestroy(graph);
        return hip_fail(e, "hipGraphInstantiate");
    }
    fh_graph* g = new (std::nothrow) fh_graph();
    if (g == nullptr) {
        (void)hipGraphExecDestroy(exec);
        (void)hipGraphDestroy(graph);
        return fail(FH_ERR_ALLOCATION, "out of host memory");
    }
    g->device = device;
    ++device->handles;
    ++device->live_graphs;
    g->graph = graph;
    g->exec = exec;
    *out = g;
    return FH_OK;
}

fh_status fh_graph_launch(fh_graph* graph) {
    if (graph == nullptr) return fail(FH_ERR_PARAMETER, "null graph");
    if (graph->device->closed) return fail(FH_ERR_DEVICE_MISMATCH, "the graph's device has been destroyed");
    if (graph->device->capturing) return fail(FH_ERR_DISPATCH, "cannot replay while recording");
    FH_HIP(hipGraphLaunch(graph->exec, graph->device->stream));
    return FH_OK;
}

void fh_graph_destroy(fh_graph* graph) {
    if (graph == nullptr) return;
    if (!graph->device->closed && graph->device->capturing) {
        graph->device->deferred_graphs.emplace_back(graph->exec, graph->graph);
    } else {
        if (!graph->device->closed) (void)hipStreamSynchronize(graph->device->stream);
        (void)hipGraphExecDestroy(graph->exec);
        (void)hipGraphDestroy(graph->graph);
    }
    if (--graph->device->live_graphs == 0 && !graph->device->capturing) {
        // nothing can replay on the outgrown scratch blocks any more
        for (void* old : graph->device->retired_scratch) release_memory(graph->device, old);
        graph->device->retired_scratch.clear();
    }
    drop_device_handle(graph->device);
    delete graph;
}

// ---- timing ---------------------------------------------------------------------------

fh_status fh_event_create(fh_device* device, fh_event** out) {
    if (device == nullptr || out == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    *out = nullptr;
    fh_event* ev = new (std::nothrow) fh_event();
    if (ev == nullptr) return fail(FH_ERR_ALLOCATION, "out of host memory");
    hipError_t e = hipEventCreate(&ev->event);
    if (e != hipSuccess) {
        delete ev;
        return hip_fail(e, "hipEventCreate");
    }
    ev->device = device;
    ++device->handles;
    *out = ev;
    return FH_OK;
}

void fh_event_destroy(fh_event* event) {
    if (event == nullptr) return;
    (void)hipEventDestroy(event->event);
    drop_device_handle(event->device);
    delete event;
}

fh_status fh_event_record(fh_event* event) {
    if (event == nullptr) return fail(FH_ERR_PARAMETER, "null event");
    if (event->device->closed) return fail(FH_ERR_DEVICE_MISMATCH, "the event's device has been destroyed");
    FH_HIP(hipEventRecord(event->event, event->device->stream));
    return FH_OK;
}

fh_status fh_event_elapsed_ms(fh_event* start, fh_event* stop, float* ms) {
    if (start == nullptr || stop == nullptr || ms == nullptr) return fail(FH_ERR_PARAMETER, "null argument");
    hipError_t e = hipEventSynchronize(stop->event);
    if (e != hipSuccess) return fail(FH_ERR_SYNCHRONIZATION, "event: %s", hipGetErrorString(e));
    FH_HIP(hipEventElapsedTime(ms, start->event, stop->event));
    return FH_OK;
}

}  // extern "C"
