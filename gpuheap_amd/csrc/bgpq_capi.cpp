// Host side of the C ABI declared in include/bgpq.h.
#include "bgpq.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "bgpq_handle.hpp"
#include "bgpq_kernels.hpp"

namespace bgpq {
const LaunchRow* rows_u32_v0();
const LaunchRow* rows_u32_v1();
const LaunchRow* rows_u32_v2();
const LaunchRow* rows_u32_v3();
const LaunchRow* rows_u64_v0();
const LaunchRow* rows_u64_v1();
const LaunchRow* rows_u64_v2();
const LaunchRow* rows_u64_v3();
}  // namespace bgpq

using namespace bgpq;

static thread_local std::string g_err;

int bgpq_fail(int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}
#define fail bgpq_fail
#define HIPCHK BGPQ_HIPCHK

static size_t key_bytes(int key_type) { return key_type == BGPQ_KEY_U64 ? 8 : 4; }

static const LaunchRow* rows_for(int key_type, int variant) {
    if (key_type == BGPQ_KEY_U32) {
        switch (variant) {
            case 0: return rows_u32_v0();
            case 1: return rows_u32_v1();
            case 2: return rows_u32_v2();
            case 3: return rows_u32_v3();
        }
    } else if (key_type == BGPQ_KEY_U64) {
        switch (variant) {
            case 0: return rows_u64_v0();
            case 1: return rows_u64_v1();
            case 2: return rows_u64_v2();
            case 3: return rows_u64_v3();
        }
    }
    return nullptr;
}

// Status words and counters sit kWordStride ints apart (one 128-byte line each).
static size_t status_bytes(int batch_num) { return sizeof(int) * kWordStride * (size_t)(batch_num + 1); }
static size_t ctr_bytes() { return sizeof(int) * kWordStride * CTR_WORDS; }

static HeapArgs args_of(const bgpq_heap* h, long long out_cap = 0) {
    return HeapArgs{h->items, h->status, h->ctr, h->init_limits, h->batch_num, 1, out_cap, nullptr};
}

// The bulk calls' words lie in the same allocations: the plan behind the
// counters, in their page, the lookback and sort words behind the slots.  (With
// the sort words behind the counters, the heap's small allocations took eight
// pages where they took six, the counters came to lie elsewhere, and single
// calls took up to 1 us longer: 54.2, 53.3, 54.2, 53.3 us an insertion into
// six heaps made in turn before, 54.5 into each of them then, 64 batches of
// 2048 u64 keys.)  Lookback words are there for the most tiles a bulk sort can
// have: of keys that take half the slots.
static size_t items_bytes(const bgpq_heap* h) {
    return key_bytes(h->key_type) * (size_t)h->batch_size * (size_t)(h->batch_num + 1);
}
static size_t up256(size_t x) { return (x + 255) & ~(size_t)255; }
static int bulk_tiles_max(const bgpq_heap* h) {
    const long long tile = h->key_type == BGPQ_KEY_U64 ? bulk_tile<uint64_t>() : bulk_tile<uint32_t>();
    const long long keys = std::min<long long>((long long)(h->batch_num + 1) * h->batch_size / 2, kBulkMaxKeys);
    return (int)(keys / tile + 1);
}
static_assert(sizeof(BulkPlan) % 4 == 0, "cleared in words");
static size_t plan_bytes() { return up256(ctr_bytes()) + sizeof(BulkPlan); }  // counters and plan
static size_t bulk_look_bytes(const bgpq_heap* h) { return sizeof(unsigned) * kRadix * (size_t)bulk_tiles_max(h); }
static size_t bulk_sort_bytes() { return sizeof(unsigned) * kSortWords; }
static void set_bulk_mem(bgpq_heap* h, bool sorts) {
    h->bulk = BulkMem{};
    h->bulk.plan = (BulkPlan*)((char*)h->ctr + up256(ctr_bytes()));
    if (!sorts) return;
    char* const p = (char*)h->items + up256(items_bytes(h));
    h->bulk.look[0] = (unsigned*)p;
    h->bulk.look[1] = (unsigned*)(p + bulk_look_bytes(h));
    h->bulk.hist = (unsigned*)(p + 2 * bulk_look_bytes(h));
    h->bulk.ticket = h->bulk.hist + kMaxPasses * kRadix;
    h->bulk.sync = (int*)(h->bulk.ticket + kMaxPasses);
    h->bulk.tiles_max = bulk_tiles_max(h);
}

static int fill_items(bgpq_heap* h, hipStream_t s) {
    const long long n = (long long)(h->batch_num + 1) * h->batch_size;
    hipError_t e = h->key_type == BGPQ_KEY_U64 ? fill_u64(h->items, n, h->init_limits, s)
                                               : fill_u32(h->items, n, (uint32_t)h->init_limits, s);
    // a kernel for the words, too: a caller may capture a reset, and memset
    // nodes of a graph have given wrong results on later replays
    if (e == hipSuccess)
        e = zero_words(h->status, (long long)(status_bytes(h->batch_num) / 4), h->ctr, (int)(plan_bytes() / 4),
                       h->bulk.hist, h->bulk.hist ? kSortWords : 0, s);
    if (e != hipSuccess) return fail(BGPQ_EHIP, "fill: %s", hipGetErrorString(e));
    return BGPQ_OK;
}

static int counters(bgpq_heap* h, int* c) {
    std::vector<int> raw((size_t)kWordStride * CTR_WORDS);
    HIPCHK(hipMemcpy(raw.data(), h->ctr, ctr_bytes(), hipMemcpyDeviceToHost));
    for (int i = 0; i < CTR_WORDS; ++i) c[i] = raw[(size_t)i * kWordStride];
    h->held = (long long)c[CTR_BATCH_COUNT] * h->batch_size + c[CTR_PARTIAL];
    return BGPQ_OK;
}

static bool capturing(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(s, &st) != hipSuccess || st != hipStreamCaptureStatusNone;
}

// The bulk calls end for good once work may run beside them: calls on a second
// stream, captured ones, whose graph may run at any time, and kernels of the
// caller on a view.  The last bulk call is waited for.
static int end_bulk(bgpq_heap* h) {
    h->shared = true;
    if (!h->bulk_open) return BGPQ_OK;
    // also while this or another thread captures
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    const hipError_t e = hipEventSynchronize(h->bulk_done);
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (e != hipSuccess) return fail(BGPQ_EHIP, "wait for the last bulk call: %s", hipGetErrorString(e));
    h->bulk_open = false;
    return BGPQ_OK;
}

int bgpq_on_stream(bgpq_heap* h, hipStream_t s) {
    std::lock_guard<std::recursive_mutex> hold(h->lock);
    if ((h->used && s != h->stream) || capturing(s)) {
        const int rc = end_bulk(h);
        if (rc) return rc;
    }
    h->used = true;
    h->stream = s;
    h->ascends = false;
    h->route = BGPQ_ROUTE_BATCHES;
    return BGPQ_OK;
}

int bgpq_handle_counters(bgpq_heap* h, int* c) { return counters(h, c); }

HeapArgs bgpq_handle_args(const bgpq_heap* h, int heap_sort) {
    HeapArgs a = args_of(h, 0);
    a.heap_sort = heap_sort;
    return a;
}

// status words 0..count-1 gathered from the padded array
static int status_words(bgpq_heap* h, int* out, int count) {
    std::vector<int> raw((size_t)kWordStride * count);
    HIPCHK(hipMemcpy(raw.data(), h->status, sizeof(int) * raw.size(), hipMemcpyDeviceToHost));
    for (int i = 0; i < count; ++i) out[i] = raw[(size_t)i * kWordStride];
    return BGPQ_OK;
}

// checkInsertHeap restated (heap/buitdd/heap.cuh:118-172, heap/tditdd/heap.cuh:123-176):
// every status word AVAIL, each batch ascending, each child's first key >=
// its parent's last key, and, when both exist, the partial buffer ascending
// and not below the root's last key.  The first violation is reported in
// the same words, and found in the same order, as the oracle's orc_check.
template <typename K>
static int check_impl(bgpq_heap* h) {
    int c[CTR_WORDS];
    int rc = counters(h, c);
    if (rc) return rc;
    const int nb = c[CTR_BATCH_COUNT], pbs = c[CTR_PARTIAL];
    const int B = h->batch_size;
    if (c[CTR_ERROR]) return fail(0, "error flags 0x%x", c[CTR_ERROR]);
    if (nb < 0 || nb > h->batch_num) return fail(0, "batch count %d", nb);
    if (pbs < 0 || pbs >= B) return fail(0, "partial size %d", pbs);
    std::vector<K> items((size_t)(nb + 1) * B);
    std::vector<int> status(nb + 1);
    HIPCHK(hipMemcpy(items.data(), h->items, sizeof(K) * items.size(), hipMemcpyDeviceToHost));
    rc = status_words(h, status.data(), nb + 1);
    if (rc) return rc;
    const bool bu = h->variant == BGPQ_BUITDD || h->variant == BGPQ_BUITDD_NP;
    if (status[0] != 0) return fail(0, "partial batch state %d, expected AVAIL", status[0]);
    if (nb != 0 && pbs != 0) {
        if (items[(size_t)2 * B - 1] > items[0])
            return fail(0, "partial buffer below the root's last key");
        for (int i = 1; i < pbs; ++i)
            if (items[i] < items[i - 1]) return fail(0, "partial buffer not ascending at %d", i);
    }
    for (int i = 1; i <= nb; ++i) {
        if (status[i] != 0) return fail(0, "state of batch %d is %d, expected AVAIL", i, status[i]);
        if (i > 1) {
            const int p = bu ? (int)rev_idx(rev_idx((uint32_t)i) >> 1) : i / 2;
            if (items[(size_t)i * B] < items[(size_t)p * B + B - 1])
                return fail(0, "batch %d below parent %d", i, p);
        }
        for (int j = 1; j < B; ++j)
            if (items[(size_t)i * B + j] < items[(size_t)i * B + j - 1])
                return fail(0, "batch %d not ascending at %d", i, j);
    }
    return 1;
}

extern "C" {

const char* bgpq_last_error(void) { return g_err.c_str(); }

int bgpq_threads(int batch_size) {
    if (batch_index(batch_size) < 0) return fail(BGPQ_EINVAL, "batch size %d not built", batch_size);
    return threads_for(batch_size);
}

int bgpq_lds_bytes(int key_type, int batch_size) {
    if (batch_index(batch_size) < 0) return fail(BGPQ_EINVAL, "batch size %d not built", batch_size);
    if (key_type != BGPQ_KEY_U32 && key_type != BGPQ_KEY_U64) return fail(BGPQ_EINVAL, "key type %d", key_type);
    return 3 * batch_size * (int)key_bytes(key_type);
}

int bgpq_default_grid(int batch_size) {
    (void)batch_size;
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 32;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        return 32;
    return cus;
}

int bgpq_create(bgpq_heap** out, int variant, int key_type, int batch_num, int batch_size,
                uint64_t init_limits) {
    if (!out) return fail(BGPQ_EINVAL, "null handle pointer");
    *out = nullptr;
    if (variant < 0 || variant > 3) return fail(BGPQ_EINVAL, "variant %d", variant);
    if (key_type != BGPQ_KEY_U32 && key_type != BGPQ_KEY_U64) return fail(BGPQ_EINVAL, "key type %d", key_type);
    const int bi = batch_index(batch_size);
    if (bi < 0) return fail(BGPQ_EINVAL, "batch size %d (need a power of two in [64, 8192])", batch_size);
    if (rows_for(key_type, variant)[bi].batch_size == 0)
        return fail(BGPQ_EINVAL, "batch size %d: %d bytes of LDS per workgroup exceed %d", batch_size,
                    3 * batch_size * (int)key_bytes(key_type), kMaxLdsBytes);
    if (batch_num < 1) return fail(BGPQ_EINVAL, "batch_num %d", batch_num);
    if (key_type == BGPQ_KEY_U32 && init_limits > 0xFFFFFFFFull)
        return fail(BGPQ_EINVAL, "init_limits does not fit u32");
    bgpq_heap* h = new bgpq_heap();
    h->variant = variant;
    h->key_type = key_type;
    h->batch_num = batch_num;
    h->batch_size = batch_size;
    h->init_limits = init_limits;
    h->row = &rows_for(key_type, variant)[bi];
    h->cus = bgpq_default_grid(batch_size);
    // A device that has no room for the lookback words (up to half a gigabyte)
    // beside the slots: the heap goes without them and without bulk calls.
    size_t bytes = 0;
    hipError_t e = hipSuccess;
    for (const bool bulk : {true, false}) {
        bytes = items_bytes(h);
        if (bulk) bytes = up256(bytes) + 2 * bulk_look_bytes(h) + bulk_sort_bytes();
        e = hipMalloc(&h->items, bytes);
        if (e == hipSuccess) e = hipMalloc((void**)&h->status, status_bytes(batch_num));
        if (e == hipSuccess) e = hipMalloc((void**)&h->ctr, plan_bytes());
        if (e == hipSuccess) {
            set_bulk_mem(h, bulk);
            break;
        }
        if (h->items) (void)hipFree(h->items);
        if (h->status) (void)hipFree(h->status);
        h->items = nullptr;
        h->status = nullptr;
    }
    if (e != hipSuccess) {
        bgpq_destroy(h);
        return fail(BGPQ_EHIP, "hipMalloc(%zu): %s", bytes, hipGetErrorString(e));
    }
    int rc = fill_items(h, nullptr);
    if (rc == BGPQ_OK && hipStreamSynchronize(nullptr) != hipSuccess) rc = fail(BGPQ_EHIP, "sync after fill");
    if (rc != BGPQ_OK) {
        bgpq_destroy(h);
        return rc;
    }
    *out = h;
    return BGPQ_OK;
}

void bgpq_destroy(bgpq_heap* h) {
    if (!h) return;
    if (h->items) (void)hipFree(h->items);
    if (h->status) (void)hipFree(h->status);
    if (h->ctr) (void)hipFree(h->ctr);
    if (h->app_ctl) (void)hipFree(h->app_ctl);
    if (h->bulk_done) (void)hipEventDestroy(h->bulk_done);
    for (hipEvent_t e : h->sort_events)
        if (e) (void)hipEventDestroy(e);
    if (h->sort_report) (void)hipHostFree(h->sort_report);
    delete h;
}

int bgpq_reset(bgpq_heap* h, void* stream) {
    if (!h) return fail(BGPQ_EINVAL, "null handle");
    std::lock_guard<std::recursive_mutex> hold(h->lock);
    const int rc = bgpq_on_stream(h, (hipStream_t)stream);
    if (rc) return rc;
    h->held = 0;
    return fill_items(h, (hipStream_t)stream);
}

int bgpq_view(bgpq_heap* h, bgpq_view_t* out) {
    if (!h || !out) return fail(BGPQ_EINVAL, "null argument");
    std::lock_guard<std::recursive_mutex> hold(h->lock);
    const int rc = end_bulk(h);
    if (rc) return rc;
    out->items = h->items;
    out->status = h->status;
    out->ctr = h->ctr;
    out->init_limits = h->init_limits;
    out->batch_num = h->batch_num;
    out->batch_size = h->batch_size;
    out->variant = h->variant;
    out->key_type = h->key_type;
    out->word_stride = kWordStride;
    out->reserved = 0;
    return BGPQ_OK;
}

int bgpq_vote_reset(bgpq_heap* h, int busy, void* stream) {
    if (!h || busy < 0) return fail(BGPQ_EINVAL, "bad vote reset");
    const int w[2] = {busy, 0};
    hipStream_t s = (hipStream_t)stream;
    const int rc = bgpq_on_stream(h, s);
    if (rc) return rc;
    HIPCHK(hipMemcpyAsync(h->ctr + CTR_BUSY * kWordStride, &w[0], sizeof(int), hipMemcpyHostToDevice, s));
    HIPCHK(hipMemcpyAsync(h->ctr + CTR_TERM * kWordStride, &w[1], sizeof(int), hipMemcpyHostToDevice, s));
    HIPCHK(hipStreamSynchronize(s));  // the words above are on this stack
    return BGPQ_OK;
}

int bgpq_terminated(bgpq_heap* h) {
    if (!h) return fail(BGPQ_EINVAL, "null handle");
    int c[CTR_WORDS];
    const int rc = counters(h, c);
    if (rc) return rc;
    return c[CTR_TERM] != 0 ? 1 : 0;
}

int bgpq_clear(bgpq_heap* h, void* stream) {
    if (!h) return fail(BGPQ_EINVAL, "null handle");
    hipStream_t s = (hipStream_t)stream;
    std::lock_guard<std::recursive_mutex> hold(h->lock);
    const int rc = bgpq_on_stream(h, s);
    if (rc) return rc;
    h->held = 0;
    const hipError_t e =
        h->key_type == BGPQ_KEY_U64
            ? clear_u64(h->items, h->status, h->ctr, h->batch_num, h->batch_size, h->init_limits, s)
            : clear_u32(h->items, h->status, h->ctr, h->batch_num, h->batch_size, (uint32_t)h->init_limits, s);
    if (e != hipSuccess) return fail(BGPQ_EHIP, "clear: %s", hipGetErrorString(e));
    return BGPQ_OK;
}

int bgpq_set_cursor(bgpq_heap* h, int64_t value) {
    if (!h || value < 0 || value > 0x7FFFFFFF) return fail(BGPQ_EINVAL, "bad cursor");
    const int v = (int)value;
    HIPCHK(hipMemcpy(h->ctr + CTR_DELETE_COUNT * kWordStride, &v, sizeof v, hipMemcpyHostToDevice));
    return BGPQ_OK;
}

int bgpq_error_flags(bgpq_heap* h, int* out) {
    if (!h || !out) return fail(BGPQ_EINVAL, "null argument");
    int c[CTR_WORDS];
    const int rc = counters(h, c);
    if (rc) return rc;
    *out = c[CTR_ERROR];
    return BGPQ_OK;
}


int bgpq_item_count(bgpq_heap* h, int64_t* out) {
    if (!h || !out) return fail(BGPQ_EINVAL, "null argument");
    int c[CTR_WORDS];
    int rc = counters(h, c);
    if (rc) return rc;
    *out = (int64_t)c[CTR_PARTIAL] + (int64_t)c[CTR_BATCH_COUNT] * h->batch_size;
    return BGPQ_OK;
}

int bgpq_node_count(bgpq_heap* h, int64_t* out) {
    if (!h || !out) return fail(BGPQ_EINVAL, "null argument");
    int c[CTR_WORDS];
    int rc = counters(h, c);
    if (rc) return rc;
    *out = c[CTR_BATCH_COUNT];
    return BGPQ_OK;
}

int bgpq_is_empty(bgpq_heap* h) {
    if (!h) return fail(BGPQ_EINVAL, "null handle");
    int c[CTR_WORDS];
    int rc = counters(h, c);
    if (rc) return rc;
    return (c[CTR_PARTIAL] == 0 && c[CTR_BATCH_COUNT] == 0) ? 1 : 0;
}

int bgpq_snapshot(bgpq_heap* h, void* h_items, int* h_status, int* h_counters) {
    if (!h) return fail(BGPQ_EINVAL, "null handle");
    HIPCHK(hipDeviceSynchronize());
    if (h_items)
        HIPCHK(hipMemcpy(h_items, h->items,
                         key_bytes(h->key_type) * (size_t)h->batch_size * (size_t)(h->batch_num + 1),
                         hipMemcpyDeviceToHost));
    if (h_status) {
        const int rc = status_words(h, h_status, h->batch_num + 1);
        if (rc) return rc;
    }
    if (h_counters) {
        int c[CTR_WORDS];
        const int rc = counters(h, c);
        if (rc) return rc;
        for (int i = 0; i < kPublicCounters; ++i) h_counters[i] = c[i];
    }
    return BGPQ_OK;
}

int bgpq_check(bgpq_heap* h) {
    if (!h) return fail(BGPQ_EINVAL, "null handle");
    HIPCHK(hipDeviceSynchronize());
    return h->key_type == BGPQ_KEY_U64 ? check_impl<uint64_t>(h) : check_impl<uint32_t>(h);
}

static int device_error(bgpq_heap* h) {
    int c[CTR_WORDS];
    int rc = counters(h, c);
    if (rc) return rc;
    if (c[CTR_ERROR]) return fail(BGPQ_EHEAP, "device error flags 0x%x", c[CTR_ERROR]);
    return BGPQ_OK;
}

static int resolve_grid(const bgpq_heap* h, int grid) { return grid > 0 ? grid : h->cus; }
// Workgroups of a per-batch launch: those beyond the calls would find nothing to
// do, and starting them took 0.3 to 0.7 us of a pop and an insertion of one
// batch (72.3 -> 71.6 us, 2048 u64 keys; 101.7 -> 101.0, 4096).
static int grid_for(const bgpq_heap* h, int grid, long long calls) {
    return (int)std::min<long long>(resolve_grid(h, grid), calls);
}

static bool np_variant(const bgpq_heap* h) { return h->variant == BGPQ_BUITDD_NP || h->variant == BGPQ_TDITDD_NP; }

// Whether calls are done together (bgpq_bulk.hpp): where one after the other
// they would take longer.  An insertion takes 2 us and a pop 4 at the least
// (B = 256), whatever the grid; a bulk call takes its launches, 60 us with a
// sort, 30 with one of one tile, 20 from slots that ascend, and its passes
// over the heap's `keys` keys (u32 keys of 4 passes 15 ps each, u64 keys of 8
// passes 50 ps).
static double sort_us(const bgpq_heap* h, long long keys, bool one = false) {
    if (one && bulk_one_tile(h, keys)) return 30.0;
    return 60.0 + keys * (h->key_type == BGPQ_KEY_U64 ? 50e-6 : 15e-6);
}
static bool bulk_fits(const bgpq_heap* h, long long keys) { return keys < kBulkMaxKeys && h->bulk.tiles_max > 0; }
static bool insert_pays(const bgpq_heap* h, long long calls, long long keys) {
    return bulk_fits(h, keys) && calls * 2.0 > sort_us(h, keys, true);
}
static bool delete_pays(const bgpq_heap* h, long long calls, long long keys, bool ascends) {
    return bulk_fits(h, keys) && calls * 4.0 > (ascends ? 20.0 + keys * 5e-6 : sort_us(h, keys));
}
static bool sort_pays(const bgpq_heap* h, long long in, long long pops, long long keys) {
    return bulk_fits(h, keys) && in * 2.0 + pops * 4.0 > sort_us(h, keys, true);
}

// A grid of one workgroup keeps the calls' own order, one after the other;
// keys that are not aligned to their size only the per-batch kernels take.
static bool bulk_can(bgpq_heap* h, const void* keys, int grid, hipStream_t s) {
    if (h->shared || grid == 1 || s == hipStreamPerThread || (uintptr_t)keys % key_bytes(h->key_type) != 0)
        return false;
    return h->bulk_done || hipEventCreateWithFlags(&h->bulk_done, hipEventDisableTiming) == hipSuccess;
}

static int insert_calls(bgpq_heap* h, const void* d_keys, int64_t n, int chunk, int grid, hipStream_t s) {
    std::lock_guard<std::recursive_mutex> hold(h->lock);
    const int rc = bgpq_on_stream(h, s);
    if (rc) return rc;
    HeapArgs a = args_of(h);
    if (insert_pays(h, (n + chunk - 1) / chunk, h->held + n) && bulk_can(h, d_keys, grid, s)) {
        const hipError_t e = bulk_insert(h, d_keys, n, nullptr, 0, 0, 0, nullptr, h->cus, s);
        if (e != hipSuccess) return fail(BGPQ_EHIP, "bulk insert launch: %s", hipGetErrorString(e));
        h->bulk_open = h->ascends = true;
        h->route = bulk_one_tile(h, h->held + n) ? BGPQ_ROUTE_TILE : BGPQ_ROUTE_SORT;
        a.skip = &h->bulk.plan->go;
    } else if (n <= chunk && solo_pays(h) && bulk_can(h, d_keys, grid, s)) {
        const hipError_t e = solo_insert(h, d_keys, (int)n, s);
        if (e != hipSuccess) return fail(BGPQ_EHIP, "insert launch: %s", hipGetErrorString(e));
        h->bulk_open = true;
        h->route = BGPQ_ROUTE_SINGLE;
        a.skip = &h->bulk.plan->go;
    }
    h->held += n;
    const hipError_t e = h->row->insert(a, d_keys, n, chunk, grid_for(h, grid, (n + chunk - 1) / chunk), s);
    if (e != hipSuccess) return fail(BGPQ_EHIP, "insert launch: %s", hipGetErrorString(e));
    return BGPQ_OK;
}

static int delete_calls(bgpq_heap* h, void* d_out, int64_t out_keys, int64_t calls, int grid, hipStream_t s) {
    std::lock_guard<std::recursive_mutex> hold(h->lock);
    const bool ascends = h->ascends;
    const int rc = bgpq_on_stream(h, s);
    if (rc) return rc;
    HeapArgs a = args_of(h, out_keys);
    const long long pops = std::min<long long>(calls, (h->held + h->batch_size - 1) / h->batch_size);
    if (delete_pays(h, pops, h->held, ascends) && bulk_can(h, d_out, grid, s)) {
        const hipError_t e = bulk_delete(h, d_out, out_keys, calls, resolve_grid(h, grid), ascends,
                                         h->cus, s);
        if (e != hipSuccess) return fail(BGPQ_EHIP, "bulk delete launch: %s", hipGetErrorString(e));
        h->bulk_open = h->ascends = true;
        h->route = ascends ? BGPQ_ROUTE_COPY : BGPQ_ROUTE_SORT;
        a.skip = &h->bulk.plan->go;
    } else if (calls == 1 && solo_pays(h) && h->held >= h->batch_size && bulk_can(h, d_out, grid, s)) {
        const hipError_t e = solo_delete(h, d_out, out_keys, s);
        if (e != hipSuccess) return fail(BGPQ_EHIP, "delete launch: %s", hipGetErrorString(e));
        h->bulk_open = true;
        h->route = BGPQ_ROUTE_SINGLE;
        a.skip = &h->bulk.plan->go;
    }
    h->held = std::max<long long>(h->held - pops * h->batch_size, 0);
    const hipError_t e = h->row->del(a, d_out, calls, grid_for(h, grid, calls), s);
    if (e != hipSuccess) return fail(BGPQ_EHIP, "delete launch: %s", hipGetErrorString(e));
    return BGPQ_OK;
}

int bgpq_insert(bgpq_heap* h, const void* d_keys, int64_t n, int chunk, int grid, void* stream) {
    if (!h) return fail(BGPQ_EINVAL, "null handle");
    if (n < 0) return fail(BGPQ_EINVAL, "n %lld", (long long)n);
    if (n == 0) return BGPQ_OK;
    if (!d_keys) return fail(BGPQ_EINVAL, "null keys");
    if (chunk <= 0) chunk = h->batch_size;
    if (chunk > h->batch_size) return fail(BGPQ_EINVAL, "chunk %d > batch size %d", chunk, h->batch_size);
    if (np_variant(h) && (chunk != h->batch_size || n % h->batch_size))
        return fail(BGPQ_EINVAL, "_np variants insert full batches only (chunk %d, n %lld)", chunk, (long long)n);
    return insert_calls(h, d_keys, n, chunk, grid, (hipStream_t)stream);
}

int bgpq_delete(bgpq_heap* h, void* d_out, int64_t out_keys, int64_t calls, int grid, void* stream) {
    if (!h) return fail(BGPQ_EINVAL, "null handle");
    if (calls < 0 || out_keys < 0) return fail(BGPQ_EINVAL, "calls %lld, out_keys %lld", (long long)calls,
                                               (long long)out_keys);
    if (calls == 0) return BGPQ_OK;
    if (!d_out) return fail(BGPQ_EINVAL, "null output");
    return delete_calls(h, d_out, out_keys, calls, grid, (hipStream_t)stream);
}

int bgpq_concurrent(bgpq_heap* h, const void* d_keys, int64_t n_insert, int chunk, void* d_out, int64_t out_keys,
                    int64_t calls, int grid, void* stream) {
    if (!h) return fail(BGPQ_EINVAL, "null handle");
    if (n_insert < 0 || calls < 0) return fail(BGPQ_EINVAL, "negative size");
    if (chunk <= 0) chunk = h->batch_size;
    if (chunk > h->batch_size) return fail(BGPQ_EINVAL, "chunk %d > batch size %d", chunk, h->batch_size);
    if (np_variant(h) && (chunk != h->batch_size || n_insert % h->batch_size))
        return fail(BGPQ_EINVAL, "_np variants insert full batches only");
    grid = resolve_grid(h, grid);
    if (grid < 2) return fail(BGPQ_EINVAL, "concurrent run needs a grid of at least 2");
    if ((n_insert && !d_keys) || (calls && !d_out)) return fail(BGPQ_EINVAL, "null buffer");
    if (out_keys < 0) return fail(BGPQ_EINVAL, "out_keys %lld", (long long)out_keys);
    hipStream_t s = (hipStream_t)stream;
    std::lock_guard<std::recursive_mutex> hold(h->lock);
    const int rc = bgpq_on_stream(h, s);
    if (rc) return rc;
    HeapArgs a = args_of(h, out_keys);
    // together: the insertions first, then the pops, one of the orders that
    // the concurrent kernel may take
    const long long in = (n_insert + chunk - 1) / chunk, all = h->held + n_insert;
    const long long pops = std::min<long long>(calls, (all + h->batch_size - 1) / h->batch_size);
    if (sort_pays(h, in, pops, all) && bulk_can(h, d_keys, grid, s) && bulk_can(h, d_out, grid, s)) {
        const hipError_t e = bulk_insert(h, d_keys, n_insert, d_out, out_keys, calls, grid - grid / 2, nullptr,
                                         h->cus, s);
        if (e != hipSuccess) return fail(BGPQ_EHIP, "bulk launch: %s", hipGetErrorString(e));
        h->bulk_open = h->ascends = true;
        h->route = bulk_one_tile(h, all) ? BGPQ_ROUTE_TILE : BGPQ_ROUTE_SORT;
        a.skip = &h->bulk.plan->go;
    }
    h->held = std::max<long long>(all - pops * h->batch_size, 0);
    hipError_t e = h->row->conc(a, d_keys, n_insert, chunk, d_out, calls, grid, s);
    if (e != hipSuccess) return fail(BGPQ_EHIP, "concurrent launch: %s", hipGetErrorString(e));
    return BGPQ_OK;
}

// A heap sort as one bulk call: both halves are one sort, and its last pass,
// which hands the keys out, counts as the second.  *done is false where the heap
// turned out not to be empty or is aborted: the caller goes on as if the call
// had not been made.  Nothing is asked of the device before or between (of 150
// us for 2^20 u32 keys, 60 were two copies of the counters, a memset and the
// making of events).
static int bulk_heapsort(bgpq_heap* h, const void* d_in, void* d_out, int64_t n, int64_t pops, int poppers,
                         float* ms_insert, float* ms_delete, hipStream_t s, bool* done) {
    hipEvent_t* const ev = h->sort_events;
    HIPCHK(hipEventRecord(ev[0], s));
    const hipError_t e = bulk_insert(h, d_in, n, d_out, n, pops + 1, poppers, ev[1],
                                     h->cus, s);
    if (e != hipSuccess) return fail(BGPQ_EHIP, "bulk launch: %s", hipGetErrorString(e));
    h->bulk_open = h->ascends = true;
    h->route = bulk_one_tile(h, n) ? BGPQ_ROUTE_TILE : BGPQ_ROUTE_SORT;
    HIPCHK(hipEventRecord(ev[2], s));
    const hipError_t r = bulk_report(h, h->sort_report, s);
    if (r != hipSuccess) return fail(BGPQ_EHIP, "report launch: %s", hipGetErrorString(r));
    HIPCHK(hipStreamSynchronize(s));
    *done = h->sort_report[0] != 0;
    if (!*done) return BGPQ_OK;
    float a = 0, b = 0;
    HIPCHK(hipEventElapsedTime(&a, ev[0], ev[1]));
    HIPCHK(hipEventElapsedTime(&b, ev[1], ev[2]));
    if (ms_insert) *ms_insert = a;
    if (ms_delete) *ms_delete = b;
    const int error = h->sort_report[1 + CTR_ERROR];
    if (error) return fail(BGPQ_EHEAP, "device error flags 0x%x", error);
    return BGPQ_OK;
}

int bgpq_heapsort(bgpq_heap* h, const void* d_in, void* d_out, int64_t n, int chunk, int grid_insert,
                  int grid_delete, float* ms_insert, float* ms_delete, void* stream) {
    if (!h) return fail(BGPQ_EINVAL, "null handle");
    if (n < 0 || (n > 0 && (!d_in || !d_out))) return fail(BGPQ_EINVAL, "bad buffers");
    if (n > 0x7FFFFFFF) return fail(BGPQ_EINVAL, "the heap-sort cursor is 32-bit: n <= 2^31-1");
    hipStream_t s = (hipStream_t)stream;
    if (chunk <= 0) chunk = h->batch_size;
    std::lock_guard<std::recursive_mutex> hold(h->lock);
    int rc = bgpq_on_stream(h, s);
    if (rc) return rc;
    const int64_t B = h->batch_size, in = (n + chunk - 1) / chunk, pops = (n + B - 1) / B;
    const bool fits = pops <= (int64_t)h->batch_num / 2;
    const bool whole = !np_variant(h) || n == 0 || (chunk == h->batch_size && n % B == 0);
    hipEvent_t* const ev = h->sort_events;
    for (int i = 0; i < 3; ++i)
        if (!ev[i]) HIPCHK(hipEventCreate(&ev[i]));
    if (h->held == 0 && fits && chunk <= h->batch_size && whole && sort_pays(h, in, pops, n) &&
        bulk_can(h, d_in, grid_insert, s) && bulk_can(h, d_out, grid_delete, s)) {
        if (!h->sort_report) HIPCHK(hipHostMalloc((void**)&h->sort_report, kReportWords * sizeof(int), 0));
        bool done = false;
        rc = bulk_heapsort(h, d_in, d_out, n, pops, resolve_grid(h, grid_delete), ms_insert, ms_delete, s, &done);
        if (rc || done) return rc;
    }
    int c[CTR_WORDS];
    rc = counters(h, c);
    if (rc) return rc;
    const long long items = (long long)c[CTR_BATCH_COUNT] * B + c[CTR_PARTIAL];
    if (items != 0) return fail(BGPQ_EINVAL, "heap sort needs an empty heap (%lld items)", items);
    if (!fits)
        return fail(BGPQ_EINVAL, "capacity: %lld keys need batch_num >= %lld", (long long)n,
                    (long long)(2 * ((n + B - 1) / B)));
    if (chunk > h->batch_size) return fail(BGPQ_EINVAL, "chunk %d > batch size %d", chunk, h->batch_size);
    if (!whole)
        return fail(BGPQ_EINVAL, "_np variants insert full batches only (chunk %d, n %lld)", chunk, (long long)n);
    HIPCHK(hipMemsetAsync(h->ctr + CTR_DELETE_COUNT * kWordStride, 0, sizeof(int), s));
    HIPCHK(hipEventRecord(ev[0], s));
    if (n > 0) rc = insert_calls(h, d_in, n, chunk, grid_insert, s);
    if (rc) return rc;
    HIPCHK(hipEventRecord(ev[1], s));
    if (!d_out) return fail(BGPQ_EINVAL, "null output");
    // enough calls to drain: every call removes a full batch or the partial buffer
    rc = delete_calls(h, d_out, n, pops + 1, grid_delete, s);
    if (rc) return rc;
    HIPCHK(hipEventRecord(ev[2], s));
    HIPCHK(hipEventSynchronize(ev[2]));
    float a = 0, b = 0;
    HIPCHK(hipEventElapsedTime(&a, ev[0], ev[1]));
    HIPCHK(hipEventElapsedTime(&b, ev[1], ev[2]));
    if (ms_insert) *ms_insert = a;
    if (ms_delete) *ms_delete = b;
    return device_error(h);
}

int bgpq_test_sort(int key_type, int batch_size, const void* d_in, const int* d_sizes, void* d_out,
                   uint64_t pad, int batches) {
    const int bi = batch_index(batch_size);
    const LaunchRow* rows = rows_for(key_type, 0);
    if (bi < 0 || !rows || batches < 1 || rows[bi].batch_size == 0)
        return fail(BGPQ_EINVAL, "bad primitive test arguments");
    hipError_t e = rows[bi].sort(d_in, d_sizes, d_out, pad, batches, nullptr);
    if (e != hipSuccess) return fail(BGPQ_EHIP, "sort launch: %s", hipGetErrorString(e));
    HIPCHK(hipDeviceSynchronize());
    return BGPQ_OK;
}

int bgpq_test_merge(int key_type, int batch_size, const void* d_a, const void* d_b, void* d_small, void* d_large,
                    int batches, int algo) {
    const int bi = batch_index(batch_size);
    const LaunchRow* rows = rows_for(key_type, 0);
    if (bi < 0 || !rows || batches < 1 || rows[bi].batch_size == 0 || algo < 0 || algo > 7)
        return fail(BGPQ_EINVAL, "bad primitive test arguments");
    hipError_t e = rows[bi].merge(d_a, d_b, d_small, d_large, batches, algo, nullptr);
    if (e != hipSuccess) return fail(BGPQ_EHIP, "merge launch: %s", hipGetErrorString(e));
    HIPCHK(hipDeviceSynchronize());
    return BGPQ_OK;
}

int bgpq_test_route(bgpq_heap* h, int* route, int* passes) {
    if (!h || !route) return fail(BGPQ_EINVAL, "null argument");
    std::lock_guard<std::recursive_mutex> hold(h->lock);
    HIPCHK(hipDeviceSynchronize());
    BulkPlan pl;
    HIPCHK(hipMemcpy(&pl, h->bulk.plan, sizeof pl, hipMemcpyDeviceToHost));
    *route = pl.go ? h->route : BGPQ_ROUTE_BATCHES;
    if (*route == BGPQ_ROUTE_SORT && pl.ascending) *route = BGPQ_ROUTE_COPY;
    if (passes) *passes = *route == BGPQ_ROUTE_SORT ? pl.active : 0;
    return BGPQ_OK;
}

int bgpq_dev_malloc(void** p, size_t bytes) {
    if (!p) return fail(BGPQ_EINVAL, "null pointer");
    HIPCHK(hipMalloc(p, bytes));
    return BGPQ_OK;
}
int bgpq_dev_free(void* p) {
    HIPCHK(hipFree(p));
    return BGPQ_OK;
}
int bgpq_h2d(void* dst, const void* src, size_t bytes) {
    HIPCHK(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
    return BGPQ_OK;
}
int bgpq_d2h(void* dst, const void* src, size_t bytes) {
    HIPCHK(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return BGPQ_OK;
}
int bgpq_sync(void) {
    HIPCHK(hipDeviceSynchronize());
    return BGPQ_OK;
}
int bgpq_device_name(char* buf, int len) {
    if (!buf || len <= 0) return fail(BGPQ_EINVAL, "buffer");
    hipDeviceProp_t p;
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    HIPCHK(hipGetDeviceProperties(&p, dev));
    snprintf(buf, (size_t)len, "%s (%s, %d CUs)", p.name, p.gcnArchName, p.multiProcessorCount);
    return BGPQ_OK;
}

}  // extern "C"
