// The C ABI's host code on a stand-in for the HIP runtime and the kernels:
// device memory is host memory, a launch only leaves a note.  It shows what the
// host decides where no GPU can (a device short of memory) or need (two threads).
//   capi_host counters   two threads: calls on a heap, and reads of its counters
//   capi_host memory     heaps that fill the device's memory
//   capi_host grids      workgroups of the per-batch launches, and what a heap allocates
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>

#include "bgpq_handle.hpp"

using namespace bgpq;

// ------------------------------------------------------------- HIP runtime
static size_t g_free = ~(size_t)0;  // of the device's memory
static int g_bulk = 0, g_rows = 0;  // launches
static int g_grid = 0;              // of the last per-batch one

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    if (n > g_free) return *p = nullptr, hipErrorOutOfMemory;
    size_t* const q = (size_t*)calloc(1, n + 16);
    g_free -= *q = n;
    return *p = q + 2, hipSuccess;
}
hipError_t hipFree(void* p) {
    size_t* const q = (size_t*)p - 2;
    g_free += *q;
    free(q);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
    return hipMemcpy(d, s, n, k);
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) { return memset(p, 0, sizeof *p), hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in"; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = (hipEvent_t)1, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) { return *t = 0, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    return *s = hipStreamCaptureStatusNone, hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
}

// ----------------------------------------------------------------- kernels
namespace bgpq {
static hipError_t row_insert(const HeapArgs&, const void*, long long, int, int grid, hipStream_t) {
    return ++g_rows, g_grid = grid, hipSuccess;
}
static hipError_t row_del(const HeapArgs&, void*, long long, int grid, hipStream_t) {
    return g_grid = grid, hipSuccess;
}
static hipError_t row_conc(const HeapArgs&, const void*, long long, int, void*, long long, int grid, hipStream_t) {
    return g_grid = grid, hipSuccess;
}
static const LaunchRow* rows() {
    static LaunchRow r[kNumBatchSizes];
    static const bool made = [] {
        for (int i = 0; i < kNumBatchSizes; ++i) r[i] = LaunchRow{64 << i, nullptr, nullptr, row_insert, row_del, row_conc};
        return true;
    }();
    (void)made;
    return r;
}
const LaunchRow* rows_u32_v0() { return rows(); }
const LaunchRow* rows_u32_v1() { return rows(); }
const LaunchRow* rows_u32_v2() { return rows(); }
const LaunchRow* rows_u32_v3() { return rows(); }
const LaunchRow* rows_u64_v0() { return rows(); }
const LaunchRow* rows_u64_v1() { return rows(); }
const LaunchRow* rows_u64_v2() { return rows(); }
const LaunchRow* rows_u64_v3() { return rows(); }
hipError_t fill_u32(void*, long long, uint32_t, hipStream_t) { return hipSuccess; }
hipError_t fill_u64(void*, long long, uint64_t, hipStream_t) { return hipSuccess; }
hipError_t clear_u32(void*, int*, int*, int, int, uint32_t, hipStream_t) { return hipSuccess; }
hipError_t clear_u64(void*, int*, int*, int, int, uint64_t, hipStream_t) { return hipSuccess; }
hipError_t bulk_insert(const bgpq_heap*, const void*, long long, void*, long long, long long, int, hipEvent_t, int,
                       hipStream_t) {
    return ++g_bulk, hipSuccess;
}
hipError_t bulk_delete(const bgpq_heap*, void*, long long, long long, int, bool, int, hipStream_t) {
    return hipSuccess;
}
hipError_t zero_words(int* status, long long nstatus, int* ctr, int nctr, unsigned* sort, int nsort, hipStream_t) {
    memset(status, 0, 4 * nstatus);
    memset(ctr, 0, 4 * nctr);
    if (nsort) memset(sort, 0, 4 * nsort);
    return hipSuccess;
}
hipError_t bulk_report(const bgpq_heap*, int*, hipStream_t) { return hipSuccess; }
bool bulk_one_tile(const bgpq_heap*, long long) { return false; }
bool solo_pays(const bgpq_heap*) { return true; }
hipError_t solo_insert(const bgpq_heap*, const void*, int, hipStream_t) { return hipSuccess; }
hipError_t solo_delete(const bgpq_heap*, void*, long long, hipStream_t) { return hipSuccess; }
}  // namespace bgpq

#define CHECK(x)                                                                     \
    do {                                                                             \
        if (!(x)) return printf("%s:%d: %s\n", __FILE__, __LINE__, #x), 1;           \
    } while (0)

static int counters() {
    bgpq_heap* h = nullptr;
    CHECK(bgpq_create(&h, BGPQ_BUITDD, BGPQ_KEY_U32, 64, 64, 0xFFFFFFFFu) == BGPQ_OK);
    uint32_t keys[64] = {}, out[64];
    std::thread reader([&] {
        int64_t n = 0;
        for (int i = 0; i < 2000; ++i) bgpq_item_count(h, &n);
    });
    int rc = BGPQ_OK;
    for (int i = 0; i < 2000 && rc == BGPQ_OK; ++i) {
        rc = bgpq_insert(h, keys, 64, 0, 0, nullptr);
        if (rc == BGPQ_OK) rc = bgpq_delete(h, out, 64, 1, 0, nullptr);
    }
    reader.join();
    CHECK(rc == BGPQ_OK);
    bgpq_destroy(h);
    return 0;
}

static int memory() {
    const int B = 1024, batches = 1 << 12;
    const size_t items = sizeof(uint32_t) * B * (batches + 1), status = 128 * (size_t)(batches + 1);
    uint32_t key = 0;
    for (const size_t room : {items + status + (64 << 10), items + status - 1, 2 * (items + status)}) {
        g_free = room;
        bgpq_heap* h = nullptr;
        const int rc = bgpq_create(&h, BGPQ_BUITDD, BGPQ_KEY_U32, batches, B, 0xFFFFFFFFu);
        if (room < items + status) {
            CHECK(rc == BGPQ_EHIP && !h && g_free == room);
            continue;
        }
        CHECK(rc == BGPQ_OK);
        g_bulk = g_rows = 0;
        CHECK(bgpq_insert(h, &key, 1000 * B, 0, 0, nullptr) == BGPQ_OK);
        // bulk calls only with their memory; the per-batch kernel always follows
        CHECK(g_rows == 1 && g_bulk == (room > items + status + (64 << 10)));
        bgpq_destroy(h);
        CHECK(g_free == room);
    }
    return 0;
}

static int grids() {
    const int B = 64;
    const size_t before = g_free;
    bgpq_heap* h = nullptr;
    CHECK(bgpq_create(&h, BGPQ_BUITDD, BGPQ_KEY_U32, 64, B, 0xFFFFFFFFu) == BGPQ_OK);
    // the counters' allocation stays in the one page it had without bulk calls
    CHECK(h->bulk.plan && (char*)(h->bulk.plan + 1) - (char*)h->ctr <= 4096 && g_free < before);
    uint32_t key = 0;
    for (int calls : {1, 3, 9})
        for (int grid : {0, 2, 5, 300}) {
            const int all = grid ? grid : 256;
            CHECK(bgpq_insert(h, &key, calls * B - 1, 0, grid, nullptr) == BGPQ_OK);
            CHECK(g_grid == (all < calls ? all : calls));
            CHECK(bgpq_delete(h, &key, 1 << 20, calls, grid, nullptr) == BGPQ_OK);
            CHECK(g_grid == (all < calls ? all : calls));
            if (grid == 0) continue;
            // half of a concurrent call's workgroups insert: its grid is what it says
            CHECK(bgpq_concurrent(h, &key, calls * B, 0, &key, 1 << 20, calls, grid, nullptr) == BGPQ_OK);
            CHECK(g_grid == grid);
        }
    bgpq_destroy(h);
    CHECK(g_free == before);
    return 0;
}

int main(int argc, char** argv) {
    const char* what = argc > 1 ? argv[1] : "";
    if (!strcmp(what, "counters")) return counters();
    if (!strcmp(what, "memory")) return memory();
    if (!strcmp(what, "grids")) return grids();
    return 2;
}
