// The heap handle behind the C ABI, shared by the heap entry points
// (bgpq_capi.cpp) and the application drivers (bgpq_apps.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bgpq.h"
#include "bgpq_bulk.hpp"
#include "bgpq_kernels.hpp"

struct bgpq_heap {
    int variant;
    int key_type;
    int batch_num;
    int batch_size;
    uint64_t init_limits;
    void* items;
    int* status;
    int* ctr;
    const bgpq::LaunchRow* row;
    long long* app_ctl;  // driver control words, allocated on first use
    bgpq::BulkMem bulk;  // working words of the bulk calls, behind ctr and items
    // Keys the heap holds as far as the host can tell without asking the
    // device.  It only chooses between the per-batch and the bulk kernels;
    // those act on the counters they find.
    long long held;
    // The bulk kernels need the heap to themselves.  They stay off once the
    // view was handed out (kernels of the caller may use the heap at any
    // time) or calls came on more than one stream.
    bool shared;
    bool used;           // a call was made, on `stream`
    hipStream_t stream;
    hipEvent_t bulk_done;  // end of the last bulk call, for calls on other streams
    bool bulk_open;
};

// To be called before work of the heap is put on a stream: notes the stream
// and, where the stream changes, waits for a bulk call on the last one.
int bgpq_on_stream(bgpq_heap* h, hipStream_t s);

namespace bgpq {
// The launch sequences of bgpq_bulk.hip.  A per-batch kernel with
// HeapArgs::skip = &plan->go must follow them, unless the plan cannot refuse.
// bulk_insert: n keys in, then `calls` deletions (0 for none).
hipError_t bulk_insert(const bgpq_heap* h, const void* keys, long long n, void* out, long long out_cap,
                       long long calls, int cus, hipStream_t s);
hipError_t bulk_delete(const bgpq_heap* h, void* out, long long out_cap, long long calls, int cus, hipStream_t s);
}  // namespace bgpq

// Records the message returned by bgpq_last_error and returns `code`.
int bgpq_fail(int code, const char* fmt, ...);
// Counter words (CTR_*) of the heap, copied to the host.
int bgpq_handle_counters(bgpq_heap* h, int* c);
// Kernel arguments of the heap; heap_sort = 0 hands popped batches to the
// caller's buffer instead of the heap-sort output cursor.
bgpq::HeapArgs bgpq_handle_args(const bgpq_heap* h, int heap_sort);

#define BGPQ_HIPCHK(expr)                                                                          \
    do {                                                                                           \
        hipError_t e_ = (expr);                                                                    \
        if (e_ != hipSuccess) return bgpq_fail(BGPQ_EHIP, "%s: %s", #expr, hipGetErrorString(e_)); \
    } while (0)
