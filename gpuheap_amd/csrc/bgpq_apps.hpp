// Heap consumers on gfx950: one persistent kernel per solve, every
// workgroup running the loop below against one shared u64 heap.
//
// The reference runs each application as a host relaunch loop around a
// persistent kernel (applications/sssp_longfei_new/main.cu:96-102,
// artifacts/astar/astar_main.cu:128-178, artifacts/knapsack/models_pq.cuh:
// 199-246) that polls heap counters between launches.  Here one launch runs
// the solve to completion: an exact count of outstanding keys (inserted and
// not yet fully processed) tells every workgroup when to leave.
//
// Loop of one workgroup:
//   1. expand the popped keys' children edge-parallel, up to 2B at a time: a
//      thread takes U (App::kEdges) consecutive edges, so that their loads
//      and atomics are in flight together (App::expand).  A round is a chain
//      of memory round trips, about 2 us however many edges it has; with one
//      edge a thread an A* solve of 1024^2 cells spent 22 of 68 ms in 13
//      rounds a pop.  Improving children go to a buffer in LDS;
//   2. outstanding += children - popped, and the children go into the heap:
//      B at a time when they pile up, all of them while the heap is short of
//      batches for the team; otherwise they are held for the next pop;
//   3. pop.  With half a batch of children or more, the workgroup exchanges
//      them with the root's batch: what it pops are the smallest of both and
//      the rest sifts down from the root (exchangeRoot), which usually ends
//      after a level or two, where an insertion and a deletion each walk
//      most of the tree (16 and 14 us of a loop of 72 us in that solve).
//      Fewer children wait beside a plain deleteRoot.  An App with
//      kThreshold (A*) pops only below App::threshold(), the A* forks'
//      deleteRoot (artifacts/astar/BGPQ_B/heap.cuh:260-287).  With nothing to
//      be had from the heap the workgroup goes on with its own children;
//   4. App::degree gives each key its number of children (0 when the key is
//      stale or pruned); a workgroup prefix scan moves the keys that have
//      children together and turns the degrees into offsets.
// Each heap operation stands in the loop once: the kernels are 60 to 90 KB
// of code, more than the instruction cache.
// With 1 to 3, against one edge a thread and every child inserted: A* on
// 1024^2 cells 64.3 -> 26.3 ms (B = 256, 4 workgroups), SSSP on R-MAT 2^18
// 10.3 -> 8.2 ms (B = 1024, 32), knapsack of 200 items 14.4 -> 12.4 ms (B =
// 256, 8), 60 mixed solves at once 45 -> 23 ms.
// Keys are never lost: outstanding reaches 0 only once the heap is empty
// and no workgroup holds keys (a workgroup's own children count from the
// moment its popped keys do not).  A threshold search ends instead with the
// heap's termination vote (PBS_MODEL, tditdd:282-289): every workgroup has
// found nothing below the threshold since its last pop.  The keys left in
// the heap then number exactly `outstanding`, all pruned.
#pragma once
#include "bgpq_device.hpp"
#include "bgpq_kernels.hpp"

namespace bgpq {

// Control words of a solve, each alone in a 128-byte line.
enum {
    APP_OUTSTANDING = 0,
    APP_POPPED = 1,
    APP_EXPANDED = 2,
    APP_STALE = 3,
    APP_PRUNED = 4,
    APP_PUSHED = 5,
    APP_ERROR = 6,
    APP_BEST = 7,  // knapsack incumbent
    APP_POOL = 8,  // knapsack node-pool cursor
    APP_DONE = 9,  // team members that have left the solve
    APP_WORDS = 10
};
constexpr int kCtlStride = 16;  // long longs per control word
enum { APPERR_RANGE = 1, APPERR_POOL = 2, APPERR_IDLE = 4, APPERR_HEAP = 8 };

// Polls of an idle workgroup (each about a microsecond) before it gives up
// and flags APPERR_IDLE: far above any real wait, it only bounds a fault.
constexpr long long kMaxIdlePolls = 1ll << 23;

__device__ __forceinline__ long long* ctl_word(long long* ctl, int i) { return ctl + (size_t)i * kCtlStride; }
__device__ __forceinline__ long long ctl_load(long long* ctl, int i) {
    return __hip_atomic_load(ctl_word(ctl, i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void ctl_add(long long* ctl, int i, long long v) {
    __hip_atomic_fetch_add(ctl_word(ctl, i), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void ctl_or(long long* ctl, int i, long long v) {
    __hip_atomic_fetch_or(ctl_word(ctl, i), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t u32_load(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t u32_min(uint32_t* p, uint32_t v) {
    return __hip_atomic_fetch_min(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t u32_max(uint32_t* p, uint32_t v) {
    return __hip_atomic_fetch_max(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t u64_load(const uint64_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void u64_store(uint64_t* p, uint64_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Exclusive prefix sum over the workgroup; `tmp` holds NT/64 values.
template <int NT, typename T>
__device__ __forceinline__ T wg_exclusive_scan(T v, T* tmp, T& total) {
    const int lane = (int)__lane_id(), wid = (int)threadIdx.x / 64;
    T x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const T y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) tmp[wid] = x;
    __syncthreads();
    T before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
        if (w == wid) before = all;
        all += tmp[w];
    }
    total = all;
    __syncthreads();
    return x - v + before;
}

// Dynamic LDS of a driver kernel, in ints: popped[B] and emit[4B] u64 keys
// (fewer than two batches are held, and a round adds two at most), off[B + 4]
// and aux[B] ints, then the heap workspace (3B keys) at app_ws_offset.
template <int B>
constexpr int app_ws_offset() { return 2 * B + 8 * B + (B + 4) + B; }
template <int B>
constexpr int app_lds_bytes() { return (app_ws_offset<B>() + 6 * B) * 4; }

// Statistics a thread gathers, added to the control words once.
struct AppStats {
    int expanded = 0, stale = 0, pruned = 0;
};

// Whether a workgroup keeps its n children for its next pops instead of
// inserting them: not while the team's other workgroups could run short of
// batches.  (Kept from a quarter, half, one or two batches for each
// workgroup on, an A* solve of 1024^2 cells by 4 took 26.4, 26.9, 28.3 and
// 36 ms, SSSP on 2^18 vertices by 32 took 8.2, 8.2, 8.4 and 10 ms.)
__device__ __forceinline__ bool keep_children(int n, int nb, int team) {
    return n == 0 || team == 1 || 4 * nb >= team;
}

// One workgroup's part in a solve.  `team` workgroups run it on the same heap
// and control words; the one with `first` set brings the first key, which the
// outstanding count already includes.
template <int VAR, int B, int NT, class App>
__device__ void drive(HeapView<uint64_t> h, const App& app, long long* ctl, uint64_t first_key, bool first,
                      int team) {
    using K = uint64_t;
    static_assert(NT <= B && B % NT == 0, "workgroup shape");
    constexpr int P = B / NT;
    constexpr int U = 2 * P < App::kEdges ? 2 * P : App::kEdges;  // edges of a thread in a round
    constexpr int kWs = app_ws_offset<B>();
    static_assert(kWs % 4 == 0, "heap workspace offset must be 16-byte aligned");
    extern __shared__ __align__(16) int app_lds[];
    K* popped = reinterpret_cast<K*>(app_lds);
    K* emit = popped + B;
    int* off = reinterpret_cast<int*>(emit + 4 * B);
    int* aux = off + B + 4;
    __shared__ int s_n, s_nb, s_part, s_any, s_done;
    __shared__ unsigned long long s_scan[NT / 64];
    DevHeap<K, VAR, B, NT> hp{h};
    constexpr bool kThr = App::kThreshold;
    const int t = threadIdx.x;
    AppStats st;
    int n_popped = 0, n_pushed = first ? 1 : 0;  // thread 0
    long long uncounted = 0, idle = 0;           // thread 0: children not yet in the outstanding count
    int n = first ? 1 : 0;                       // children held, in emit[0 .. n)
    int size = 0, total = 0, active = 0;         // keys popped, their children, the keys that have any
    if (t == 0) {
        bcast_slots()[BC_ABORT] = 0;
        s_n = n;
        if (first) emit[0] = first_key;
    }
    app.stage();
    __syncthreads();
    if (kThr && first) hp.voteBusy();  // counted busy by the solve's setup
    while (!hp.aborted()) {
        // ---- expand the popped keys' children
        int e0 = 0, nb = 0, part = 0;
        bool any = false;
        do {
            if (e0 < total) {
                const int e = e0 + t * U;
                K parent[U], child[U];
                int j[U], ax[U];
                bool ok[U];
                int lo = 0;  // the last key with off <= e
                if constexpr (App::kChildren > 0) {
                    lo = e < total ? e / App::kChildren : 0;
                } else {
                    int hi = active - 1;
                    while (lo < hi) {
                        const int mid = (lo + hi + 1) >> 1;
                        if (off[mid] <= e) lo = mid;
                        else hi = mid - 1;
                    }
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    ok[u] = e + u < total;
                    if (u > 0 && ok[u] && off[lo + 1] <= e + u) ++lo;  // every key here has children
                    parent[u] = popped[lo];
                    j[u] = e + u - off[lo];
                    ax[u] = aux[lo];
                }
                app.expand(parent, j, ax, ok, child);
                // a place in the buffer for each improving child, a wave at a time
                unsigned long long m[U];
                int cnt = 0;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    m[u] = __ballot(ok[u]);
                    cnt += __popcll(m[u]);
                }
                if (cnt > 0) {
                    const int lane = (int)__lane_id();
                    int at = 0;
                    if (lane == 0) at = atomicAdd(&s_n, cnt);
                    at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        if (ok[u]) emit[at + __popcll(m[u] & ((1ull << lane) - 1))] = child[u];
                        at += __popcll(m[u]);
                    }
                }
            }
            e0 += NT * U;
            __syncthreads();
            const int held = n;
            const bool done = e0 >= total;
            n = s_n;
            if (t == 0) {
                uncounted += n - held;
                n_pushed += n - held;
                if (done || n >= 2 * B) {
                    // children count before others can meet them; the popped
                    // keys leave the count once all their children are in it
                    const long long d = uncounted - (done ? size : 0);
                    if (d != 0) ctl_add(ctl, APP_OUTSTANDING, d);
                    uncounted = 0;
                    if (done) {
                        const int batches = a_load(h.ctr + CTR_BATCH_COUNT * kWordStride);
                        const int part = a_load(h.ctr + CTR_PARTIAL * kWordStride);
                        s_nb = batches;
                        s_part = part;
                        // a busy workgroup must reach deleteRoot to cast its idle vote
                        s_any = (batches | part) != 0 || (kThr && hp.busy_);
                    }
                    wait_stores();
                }
            }
            __syncthreads();
            // ---- into the heap: whole batches when they pile up; after the
            // last round everything that is not kept for the next pop
            bool all = false;
            if (done) {
                nb = s_nb;
                part = s_part;
                any = s_any != 0;
                all = !keep_children(n, nb, team);
            }
            while (n >= 2 * B || (all && n > 0)) {
                const int m = n < B ? n : B;
                n -= m;
                hp.insertion(emit + n, m, kWs);
                if (hp.aborted()) break;
                any = true;
                __syncthreads();
                if (t == 0) s_n = n;
                __syncthreads();
            }
        } while (e0 < total && !hp.aborted());
        if (hp.aborted()) break;
        // ---- pop: enough children are exchanged with the root's batch; a few
        // wait for more, and are all there is to go on with once the heap has
        // nothing to hand out
        int from = 0, m = 0;  // the popped keys: popped[from .. from + size)
        bool sift = false;
        size = total = 0;
        if (n >= B / 2 && nb > 0) {
            if (part > 0) n += hp.takePartial(emit + n);
            m = n < B ? n : B;
            sift = hp.exchangeRoot(emit, m, popped, kWs);
            if (sift) from = B - m;
        } else if (any) {
            if (t == 0) hp.hold_ = n;
            if constexpr (kThr) sift = hp.deleteRoot(popped, size, app.threshold(), kWs);
            else sift = hp.deleteRoot(popped, size, kWs);
        }
        if (hp.aborted()) break;
        if (n > 0 && size == 0) {
            // the first m children were exchanged, or are popped themselves;
            // the rest moves up by m = B places, up to 2B of them where the
            // partial buffer's keys came in
            m = n < B ? n : B;
            if (!sift)
                for (int i = t; i < m; i += NT) popped[i] = emit[i];
            size = m;
            n -= m;
            for (int i = t; i < n; i += NT) emit[i] = emit[B + i];  // a thread reads each place before it writes it
            if (t == 0) s_n = n;
        }
        if (sift) hp.deleteUpdate(kWs);
        if (hp.aborted()) break;
        if (size == 0) {
            // (a word of its own: with nothing to be had there was no barrier
            // since s_any was read)
            if (t == 0) {
                bool over = kThr ? a_load(h.ctr + CTR_TERM * kWordStride) != 0 : ctl_load(ctl, APP_OUTSTANDING) == 0;
                if (!over && ++idle > kMaxIdlePolls) {
                    ctl_or(ctl, APP_ERROR, APPERR_IDLE);
                    over = true;
                }
                s_done = over;
            }
            __syncthreads();
            const bool done = s_done != 0;
            __syncthreads();
            if (done) break;
            backoff();
            continue;
        }
        idle = 0;
        __syncthreads();
        // ---- degrees; the keys that have children move together, with their offsets
        K key[P];
        int deg[P], extra[P];
        unsigned long long sum = 0;  // keys with children << 32 | children
#pragma unroll
        for (int p = 0; p < P; ++p) key[p] = popped[from + (t * P + p < size ? t * P + p : 0)];
        app.degree(key, size - t * P, deg, extra, st);  // key: what expand is to get
#pragma unroll
        for (int p = 0; p < P; ++p) sum += deg[p] > 0 ? (1ull << 32) + (unsigned)deg[p] : 0ull;
        unsigned long long sums = 0;
        unsigned long long pre = wg_exclusive_scan<NT>(sum, s_scan, sums);
        total = (int)(unsigned)sums;
        active = (int)(sums >> 32);
#pragma unroll
        for (int p = 0; p < P; ++p) {
            if (deg[p] > 0) {
                const int i = (int)(pre >> 32);
                popped[i] = key[p];
                off[i] = (int)(unsigned)pre;
                aux[i] = extra[p];
                pre += (1ull << 32) + (unsigned)deg[p];
            }
        }
        if (t == 0) {
            off[active] = total;
            n_popped += size;
        }
        __syncthreads();
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        st.expanded += __shfl_xor(st.expanded, o, 64);
        st.stale += __shfl_xor(st.stale, o, 64);
        st.pruned += __shfl_xor(st.pruned, o, 64);
    }
    if (__lane_id() == 0) {
        ctl_add(ctl, APP_EXPANDED, st.expanded);
        ctl_add(ctl, APP_STALE, st.stale);
        ctl_add(ctl, APP_PRUNED, st.pruned);
    }
    __syncthreads();
    if (t == 0) {
        if (hp.aborted()) ctl_or(ctl, APP_ERROR, APPERR_HEAP);
        ctl_add(ctl, APP_POPPED, n_popped);
        ctl_add(ctl, APP_PUSHED, n_pushed);
    }
}

// ------------------------------------------------------------------ SSSP
// Keys dist << 32 | vertex (applications/sssp_longfei_new/sssp.cu:6).  A key
// whose dist is above the vertex's current label is stale (sssp.cu:48-57);
// relaxations use atomicMin on the labels (sssp.cu:103-120).
struct SsspApp {
    static constexpr bool kThreshold = false;
    static constexpr int kEdges = 4;     // a thread expands at once
    static constexpr int kChildren = 0;  // of every key that has any (0: they differ)
    const int* rowptr;
    const int* col;
    const uint32_t* w;
    uint32_t* dist;
    long long* ctl;
    __device__ void stage() const {}
    // Children of the first `in` keys (0 for the others, which repeat a
    // valid key); `extra`: the vertex's first edge.
    template <int P>
    __device__ void degree(uint64_t (&key)[P], int in, int (&deg)[P], int (&extra)[P], AppStats& st) const {
        uint32_t label[P];
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const uint32_t v = (uint32_t)key[i];
            extra[i] = rowptr[v];
            deg[i] = rowptr[v + 1];
            label[i] = u32_load(dist + v);
        }
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const bool live = (uint32_t)(key[i] >> 32) <= label[i];
            st.stale += i < in && !live;
            st.expanded += i < in && live;
            deg[i] = i < in && live ? deg[i] - extra[i] : 0;
        }
    }
    template <int U>
    __device__ void expand(const uint64_t (&key)[U], const int (&j)[U], const int (&extra)[U], bool (&ok)[U],
                           uint64_t (&child)[U]) const {
        uint32_t u[U], wt[U], label[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const int idx = ok[i] ? extra[i] + j[i] : extra[0];
            u[i] = (uint32_t)col[idx];
            wt[i] = w[idx];
        }
#pragma unroll
        for (int i = 0; i < U; ++i) label[i] = u32_load(dist + u[i]);
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const uint64_t nd = (key[i] >> 32) + wt[i];
            if (ok[i] && nd >= 0xFFFFFFFFull) ctl_or(ctl, APP_ERROR, APPERR_RANGE);
            ok[i] = ok[i] && nd < 0xFFFFFFFFull && nd < label[i];
            child[i] = nd << 32 | u[i];
        }
#pragma unroll
        for (int i = 0; i < U; ++i)
            if (ok[i]) label[i] = u32_min(dist + u[i], (uint32_t)(child[i] >> 32));
#pragma unroll
        for (int i = 0; i < U; ++i) ok[i] = ok[i] && (uint32_t)(child[i] >> 32) < label[i];
    }
};

// -------------------------------------------------------------------- A*
// Keys f << 32 | cell on an 8-connected grid; moves cost 10 / 14 into any
// free cell (artifacts/astar/pq_model.cuh:114-184 checks only the target
// cell), octile heuristic.  Pops stop at the goal's label: deleteRoot with
// the threshold g[goal] << 32 hands out only keys whose f is below it (the
// reference passes dist[target], pq_model.cuh:287-296, to
// artifacts/astar/BGPQ_B/heap.cuh:273-287).  A popped key whose g is above
// the cell's label is stale; one whose f has reached the goal's label since
// it was popped is pruned.
struct AstarApp {
    static constexpr bool kThreshold = true;
    static constexpr int kEdges = 4;
    static constexpr int kChildren = 8;
    const uint8_t* free_cells;
    int width, height;
    uint32_t* g;
    long long* ctl;
    // octile distance from (x, y) to the goal
    __device__ uint32_t h(int x, int y) const {
        const uint32_t dx = (uint32_t)(width - 1 - x), dy = (uint32_t)(height - 1 - y);
        const uint32_t lo = dx < dy ? dx : dy, hi = dx < dy ? dy : dx;
        return 10u * hi + 4u * lo;
    }
    __device__ uint32_t goal() const { return (uint32_t)width * (uint32_t)height - 1u; }
    __device__ uint64_t threshold() const { return (uint64_t)u32_load(g + goal()) << 32; }
    __device__ void stage() const {}
    // `extra`: the cell's row
    template <int P>
    __device__ void degree(uint64_t (&key)[P], int in, int (&deg)[P], int (&extra)[P], AppStats& st) const {
        uint32_t label[P];
        const uint32_t best = u32_load(g + goal());
#pragma unroll
        for (int i = 0; i < P; ++i) label[i] = u32_load(g + (uint32_t)key[i]);
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const uint32_t f = (uint32_t)(key[i] >> 32), cell = (uint32_t)key[i];
            const int y = (int)(cell / (uint32_t)width);
            const bool stale = f - h((int)(cell - (uint32_t)y * (uint32_t)width), y) > label[i];
            const bool pruned = !stale && (cell == goal() || f >= best);
            st.stale += i < in && stale;
            st.pruned += i < in && pruned;
            st.expanded += i < in && !stale && !pruned;
            extra[i] = y;
            deg[i] = i < in && !stale && !pruned ? 8 : 0;
        }
    }
    template <int U>
    __device__ void expand(const uint64_t (&key)[U], const int (&j)[U], const int (&extra)[U], bool (&ok)[U],
                           uint64_t (&child)[U]) const {
        uint32_t nb[U], ng[U], nf[U], label[U], best = u32_load(g + goal());
        uint8_t open[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const uint32_t f = (uint32_t)(key[i] >> 32), cell = (uint32_t)key[i];
            const int y0 = extra[i], x0 = (int)(cell - (uint32_t)y0 * (uint32_t)width);
            const int k = j[i] < 4 ? j[i] : j[i] + 1;  // 3x3 neighbourhood without the centre
            const int dy = k / 3 - 1, dx = k - 3 * (dy + 1) - 1;
            const int x = x0 + dx, y = y0 + dy;
            ok[i] = ok[i] && x >= 0 && y >= 0 && x < width && y < height;
            nb[i] = ok[i] ? (uint32_t)y * (uint32_t)width + (uint32_t)x : 0u;
            ng[i] = f - h(x0, y0) + ((dx != 0 && dy != 0) ? 14u : 10u);
            nf[i] = ng[i] + h(x, y);
            open[i] = free_cells[nb[i]];
            label[i] = u32_load(g + nb[i]);
        }
#pragma unroll
        for (int i = 0; i < U; ++i) {
            ok[i] = ok[i] && open[i] && nf[i] < best && ng[i] < label[i];
            child[i] = (uint64_t)nf[i] << 32 | nb[i];
        }
#pragma unroll
        for (int i = 0; i < U; ++i)
            if (ok[i]) label[i] = u32_min(g + nb[i], ng[i]);
#pragma unroll
        for (int i = 0; i < U; ++i) ok[i] = ok[i] && ng[i] < label[i];
    }
};

// -------------------------------------------------------------- knapsack
// Best-first 0/1 branch-and-bound (artifacts/knapsack/knapsackKernel.cuh:
// 4-91: branch on the next item in value/weight order, bound by the
// fractional relaxation) with an integer Dantzig bound and dominance: a
// node survives only if its value beats the best recorded for its
// (depth, used weight) cell, and a popped node whose cell has since
// improved is stale.  Nodes are 16-byte records in a pool; the key's low
// word is the record index.  Every array of the solve is read with
// device-coherent loads: a long-running serving kernel may meet them in
// memory it has cached under an earlier query.
struct KnapNode {
    uint32_t level, used, value, pad;
};
constexpr uint64_t kUbTop = (1ull << 24) - 1;

__device__ __forceinline__ uint64_t knap_key(uint64_t ub, uint32_t level, uint32_t idx) {
    return ((((kUbTop - ub) << 8) | (uint64_t)(255u - level)) << 32) | idx;
}

struct KnapsackApp {
    static constexpr bool kThreshold = false;
    static constexpr int kEdges = 2;
    static constexpr int kChildren = 2;
    int n;
    uint64_t cap;
    const uint32_t* w;      // item weights in value/weight order
    const uint32_t* v;
    const uint64_t* pw;     // prefix sums of w and v, n + 1 entries
    const uint64_t* pv;
    uint32_t* cell;         // (n + 1) * (cap + 1): best value + 1
    KnapNode* pool;
    long long pool_cap;
    long long* ctl;

    // (In words: a 16-byte buffer load of a place that differs from lane to
    // lane is a loop over the lanes, 10 us for a wave's records.)
    __device__ KnapNode load_node(uint32_t idx) const {
        const uint64_t* q = reinterpret_cast<const uint64_t*>(pool + idx);
        const uint64_t a = u64_load(q), b = u64_load(q + 1);
        return KnapNode{(uint32_t)a, (uint32_t)(a >> 32), (uint32_t)b, (uint32_t)(b >> 32)};
    }
    __device__ uint32_t* slot(uint32_t level, uint64_t used) const {
        return cell + (size_t)level * (cap + 1) + used;
    }
    // The items' arrays in LDS, for the bounds' searches: read from memory (a
    // device-coherent load is a round trip of about 0.7 us) a search alone
    // took 6 us.
    struct Items {
        uint64_t pw[256];
        uint32_t pv[256], w[256], v[256];
    };
    __device__ __forceinline__ static Items& items() {
        __shared__ Items s;
        return s;
    }
    __device__ void stage() const {
        Items& s = items();
        for (int i = threadIdx.x; i <= n; i += blockDim.x) {
            s.pw[i] = u64_load(pw + i);
            s.pv[i] = (uint32_t)u64_load(pv + i);
            s.w[i] = i < n ? u32_load(w + i) : 1u;
            s.v[i] = i < n ? u32_load(v + i) : 0u;
        }
    }
    // What expand gets: the node's value in place of its record's index, and
    // the weight used (`extra`), so that it need not load the record again.
    template <int P>
    __device__ void degree(uint64_t (&key)[P], int in, int (&deg)[P], int (&extra)[P], AppStats& st) const {
        KnapNode nd[P];
        uint32_t held[P];
        const long long best = ctl_load(ctl, APP_BEST);
#pragma unroll
        for (int i = 0; i < P; ++i) nd[i] = load_node((uint32_t)key[i]);
#pragma unroll
        for (int i = 0; i < P; ++i) held[i] = u32_load(slot(nd[i].level, nd[i].used));
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const bool pruned = (long long)(kUbTop - (key[i] >> 40)) <= best || (int)nd[i].level >= n;
            const bool stale = !pruned && held[i] != nd[i].value + 1;
            st.pruned += i < in && pruned;
            st.stale += i < in && stale;
            st.expanded += i < in && !stale && !pruned;
            deg[i] = i < in && !stale && !pruned ? 2 : 0;
            key[i] = (key[i] >> 32) << 32 | nd[i].value;
            extra[i] = (int)nd[i].used;
        }
    }
    // Child 0 takes the node's item, child 1 leaves it.  The bound of a child
    // at level cl with `room` left: its value, the items from cl on while
    // they fit whole, and floor(room * v / w) of the first that does not.
    template <int U>
    __device__ void expand(const uint64_t (&key)[U], const int (&j)[U], const int (&extra)[U], bool (&ok)[U],
                           uint64_t (&child)[U]) const {
        const Items& it = items();
        uint32_t wl[U], vl[U], cl[U];
        uint32_t value[U], ub[U];  // total values lie below 2^24, weights up to cap below 2^32
        uint64_t used[U], base[U];
        long long best = ctl_load(ctl, APP_BEST);
#pragma unroll
        for (int i = 0; i < U; ++i) {
            cl[i] = 256u - ((uint32_t)(key[i] >> 32) & 255u);  // the key's level + 1
            wl[i] = it.w[cl[i] - 1];
            vl[i] = it.v[cl[i] - 1];
            base[i] = it.pw[cl[i]];
            ub[i] = it.pv[cl[i]];
        }
        long long top = 0;
#pragma unroll
        for (int i = 0; i < U; ++i) {
            used[i] = (uint64_t)(uint32_t)extra[i] + (j[i] == 0 ? wl[i] : 0u);
            value[i] = (uint32_t)key[i] + (j[i] == 0 ? vl[i] : 0u);
            ok[i] = ok[i] && used[i] <= cap;
            if (ok[i] && (long long)value[i] > top) top = (long long)value[i];
            ok[i] = ok[i] && (int)cl[i] < n;
        }
        if (top > best)
            __hip_atomic_fetch_max(ctl_word(ctl, APP_BEST), top, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // largest m with pw[m] - pw[cl] <= room, n <= 255 items: 8 halvings
        int lo[U], hi[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            lo[i] = ok[i] ? (int)cl[i] : 0;
            hi[i] = ok[i] ? n : 0;
        }
        for (int step = 0; step < 8; ++step) {
            uint64_t q[U];
#pragma unroll
            for (int i = 0; i < U; ++i) q[i] = it.pw[(lo[i] + hi[i] + 1) >> 1];
#pragma unroll
            for (int i = 0; i < U; ++i) {
                const int mid = (lo[i] + hi[i] + 1) >> 1;
                if (lo[i] < hi[i]) {
                    if (q[i] - base[i] <= cap - used[i]) lo[i] = mid;
                    else hi[i] = mid - 1;
                }
            }
        }
        uint64_t fit[U];
        uint32_t gain[U];
        best = ctl_load(ctl, APP_BEST);
#pragma unroll
        for (int i = 0; i < U; ++i) {
            fit[i] = it.pw[lo[i]];
            gain[i] = it.pv[lo[i]];
            wl[i] = it.w[lo[i]];
            vl[i] = it.v[lo[i]];
        }
        uint32_t seen[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            ub[i] = value[i] + (gain[i] - ub[i]);
            if (ok[i]) ub[i] += (uint32_t)((cap - used[i] - (fit[i] - base[i])) * vl[i] / wl[i]);
            ok[i] = ok[i] && (long long)ub[i] > best;
            if (ok[i]) seen[i] = u32_max(slot(cl[i], used[i]), value[i] + 1);
        }
        // records of the pool for what is not dominated, a wave at a time
        unsigned long long m[U];
        int cnt = 0;
#pragma unroll
        for (int i = 0; i < U; ++i) {
            ok[i] = ok[i] && value[i] + 1 > seen[i];
            m[i] = __ballot(ok[i]);
            cnt += __popcll(m[i]);
        }
        if (cnt == 0) return;
        const int first = __ffsll(__ballot(true)) - 1;
        long long at = 0;
        if ((int)__lane_id() == first)
            at = __hip_atomic_fetch_add(ctl_word(ctl, APP_POOL), (long long)cnt, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT);
        at = __shfl(at, first, 64);
        // in the edges' order: among equal bounds the lower index pops first
#pragma unroll
        for (int i = 0; i < U; ++i) at += __popcll(m[i] & ((1ull << __lane_id()) - 1));
#pragma unroll
        for (int i = 0; i < U; ++i) {
            const long long idx = at;
            at += ok[i] ? 1 : 0;
            if (ok[i] && idx >= pool_cap) {
                ctl_or(ctl, APP_ERROR, APPERR_POOL);
                ok[i] = false;
            }
            if (ok[i]) {
                uint64_t* q = reinterpret_cast<uint64_t*>(pool + idx);
                u64_store(q, (uint64_t)(uint32_t)used[i] << 32 | cl[i]);
                u64_store(q + 1, value[i]);
                child[i] = knap_key(ub[i], cl[i], (uint32_t)idx);
            }
        }
    }
};

}  // namespace bgpq
