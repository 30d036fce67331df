// The heap handle behind the C ABI, shared by the heap entry points
// (bgpq_capi.cpp) and the application drivers (bgpq_apps.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <mutex>

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
    int cus;             // compute units of its device: the default grid
    long long* app_ctl;  // driver control words, allocated on first use
    bgpq::BulkMem bulk;  // working words of the bulk calls, behind ctr and items
    // Keys the heap holds as far as the host can tell without asking the
    // device.  It only chooses between the per-batch and the bulk kernels;
    // those act on the counters they find.  Atomic: whoever reads the counters
    // (bgpq_item_count and the like) corrects it beside other threads' calls.
    std::atomic<long long> held;
    // The bulk kernels need the heap to themselves.  They stay off once the
    // view was handed out (kernels of the caller may use the heap at any
    // time) or calls came on more than one stream.
    bool shared;
    bool used;           // a call was made, on `stream`
    hipStream_t stream;
    hipEvent_t bulk_done;  // end of the last bulk call, made with the first
    bool bulk_open;        // calls on another stream have to wait for it
    bool ascends;          // like `held`: the last call was a bulk call
    int route;             // of the last call, if the plan did not refuse (bgpq_route)
    // A heap sort's start, middle and end, and what its end tells the host;
    // made with the first one.
    hipEvent_t sort_events[3];
    int* sort_report;
    // Held while a call's kernels are put on its stream: a bulk call's
    // kernels must not mix with those of another thread's call.
    std::recursive_mutex lock;
};

// To be called before work of the heap is put on a stream: notes the stream
// and, where it changes or is captured, ends the bulk calls and waits for the
// last one.
int bgpq_on_stream(bgpq_heap* h, hipStream_t s);

namespace bgpq {
// The launch sequences of bgpq_bulk.hip.  A per-batch kernel with
// HeapArgs::skip = &plan->go must follow them, unless the plan cannot refuse.
// bulk_insert: n keys in, then `calls` deletions (0 for none), which count in
// the termination vote as those of `poppers` workgroups.  With `mid` a
// heap sort: refused unless the heap is empty, the output starts at its first
// key whatever the cursor, and `mid` is recorded before the pass that hands
// the keys out (before the one kernel of a sort of one tile).
// bulk_report: kReportWords words of pinned memory, behind a heap sort.
// bulk_delete: `ascends` where the slots are expected to ascend (a plan that
// finds otherwise refuses).
hipError_t bulk_insert(const bgpq_heap* h, const void* keys, long long n, void* out, long long out_cap,
                       long long calls, int poppers, hipEvent_t mid, int cus, hipStream_t s);
// Whether an insertion that makes `keys` keys in all is sorted by one workgroup.
bool bulk_one_tile(const bgpq_heap* h, long long keys);
hipError_t bulk_report(const bgpq_heap* h, int* report, hipStream_t s);
hipError_t bulk_delete(const bgpq_heap* h, void* out, long long out_cap, long long calls, int poppers, bool ascends,
                       int cus, hipStream_t s);
// A heap's status words, counters and plan, and sort words to 0.
hipError_t zero_words(int* status, long long nstatus, int* ctr, int nctr, unsigned* sort, int nsort, hipStream_t s);
// bgpq_solo.hip: one insertion of `size` keys, one pop; like bulk calls, with
// plan->go.  solo_pays: the batch sizes where they are the faster ones.
bool solo_pays(const bgpq_heap* h);
hipError_t solo_insert(const bgpq_heap* h, const void* keys, int size, hipStream_t s);
hipError_t solo_delete(const bgpq_heap* h, void* out, long long out_cap, hipStream_t s);
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
