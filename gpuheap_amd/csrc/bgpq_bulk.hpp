// Bulk insertion and bulk deletion: the calls that carry many batches.
//
// One insertion or deletion after the other meets every other one at the
// root, and that chain of lock hand-offs bounds the per-batch kernels (about
// 3 us per insertion and 4.4 us per pop at B = 1024 u32 whatever the grid,
// 3% of HBM bandwidth).  A call with many batches does not need that order:
// the heap after n insertions may be any valid heap over the same keys, and
// k pops hand out the k * B smallest keys in ascending order.  So such a call
// sorts the heap's keys (and the new ones) with a device-wide radix sort and
// lays them out again as a heap whose slots ascend, which every variant
// accepts: a slot's parent is always a lower slot, the partial buffer takes
// the largest keys.
//
// The heap is quiescent while these kernels run (a call is ordered on its
// stream), and every status word stays AVAIL.  No memory is allocated: the
// sort's second buffer is the heap's own free slots, which are filled with
// init_limits again afterwards; a heap too full for that takes the per-batch
// path.  What the call does is decided on the device from the heap's
// counters (BulkPlan), so nothing waits for the host.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bgpq {

constexpr int kRadix = 256;        // 8-bit digits
constexpr int kMaxPasses = 8;      // of a u64 key
constexpr int kBulkThreads = 512;  // of a pass's workgroup (8 waves)
// Keys a workgroup takes at a time (a tile): 32 or 64 KB of LDS, which with the
// counters leave room for 3 and 2 workgroups on a CU.  Large tiles have fewer
// look-backs and longer runs to write, but a small sort waits longer for its
// one round of tiles.  They are the faster ones from large_tiles_from keys on
// (heap sorts, 32 and 64 KB: u32 keys, 2^20 101 and 113 us, 2^22 172 and 163,
// 2^24 324 and 301, 2^26 1067 and 918; u64 keys, 300,000 125 and 157, 1 M 161
// and 163, 1.5 M 196 and 186, 3 M 258 and 238).  Tiles below 32 KB are no
// faster even where they would reach more CUs, since the look-back gets longer
// (2^20 u32 keys: 159, 163, 182 us with 32, 16, 8 KB; rounds of 1.5 M u64 keys
// in all: 983, 1103, 1415 us).
template <typename K>
constexpr int bulk_tile(bool large = false) { return (large ? 65536 : 32768) / (int)sizeof(K); }
template <typename K>
constexpr long long large_tiles_from() { return sizeof(K) == 4 ? 1ll << 22 : 1500000; }
// Above this the lookback words' 30-bit counts would not do.
constexpr long long kBulkMaxKeys = 1ll << 30;

// What a bulk call does, decided by plan_insert or k_plan_delete.
struct BulkPlan {
    int go;               // 0: the per-batch kernel runs instead
    int ascending;        // delete: the slots already ascend, no sort needed
    int drains;           // every key is handed out
    int nb, pbs;          // batches and partial keys found
    int total;            // keys sorted
    int tiles;
    int cut;              // keys handed out, the smallest `cut`
    int off;              // where they start in the output
    int nb_after, pbs_after;
    int full_after;       // nb_after * B
    long long spare;      // first key index of the free slots used
    long long fill_lo, fill_hi;  // key range refilled with init_limits
    int error;            // error flags to raise
    // termination vote: deletions that found nothing, and workgroups left busy
    int idle, busy;
    int active;           // passes that move keys: the last launches
    int order[kMaxPasses];  // of a launch: its pass's position << 8 | its digit, -1: none
    int through_out;        // the passes alternate between the free slots and the output
};

// Device memory of a handle's bulk calls.  The sort words (hist, ticket,
// sync) are 0 between calls.
struct BulkMem {
    BulkPlan* plan;
    unsigned* hist;      // [kMaxPasses][kRadix] key counts, then first positions
    unsigned* ticket;    // [kMaxPasses] next tile of a pass
    int* sync;           // violations found, workgroups arrived
    unsigned* look[2];   // [tiles][kRadix] lookback words, alternating by pass
    int tiles_max;
};
// What a heap sort's end tells the host (pinned memory): the plan's `go` and
// the counter words.
constexpr int kReportWords = 16;
constexpr int kSortWords = kMaxPasses * (kRadix + 1) + 2;

// One bulk call on one heap.
template <typename K>
struct BulkArgs {
    K* items;
    int* ctr;
    K init_limits;
    int batch_num, batch_size;
    const K* keys;  // inserted
    long long n;
    K* out;         // popped, by `calls` deletions
    long long out_cap, calls;
    int poppers;    // workgroups that would pop them one after the other (the vote counts them)
    int tile;       // keys of a tile
    int from_empty; // only on an empty heap, the output from its start
    int planned;    // the plan is in memory already (k_plan_delete)
    int sorts;      // the sort's kernels follow, not the copy of ascending slots
    BulkMem mem;
};

}  // namespace bgpq
