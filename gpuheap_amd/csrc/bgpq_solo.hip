// One insertion or one pop on a heap that has itself to itself (bgpq_handle.hpp:
// the condition of the bulk calls): one workgroup, no locks.
//
// A single call is a chain of levels, 12 of them for 4096 batches, and a level
// of the shared heap's walk is a chain of round trips to memory: the locks,
// the batches, the stores before the release (about 3 us).  Alone, the walk
// needs neither the locks nor the waits for its stores, and the batches of the
// levels to come are loaded while the present one is merged: an insertion's
// path is known from its slot, a pop's next level once its children have been
// compared.
//
// One insertion and one pop, 1024 batches held, the host's part and the wait
// included (us; shared kernels, here):
//   u32  B = 64    37 and 39, 23 and 26      u64  B = 64   39 and 41, 26 and 28
//        256       40 and 43, 25 and 28           256      46 and 51, 31 and 34
//        1024      45 and 44, 32 and 36           512      53 and 56, 38 and 42
//        4096      57 and 56, 46 and 47           1024     59 and 53, 57 and 62
// u64 keys from B = 1024 on, where the shared sift takes its merges by halves,
// and u32 keys of B = 8192 stay with the shared kernels (solo_pays; beyond that
// line B = 2048 u64 has 67 and 64, 62 and 61, and 8192 u32 77 and 75, 72 and 67).
//
// The heap that is left is one that any order of calls could have left: the
// same counters, every status word AVAIL, free slots at init_limits.  A call
// that finds the heap otherwise than it needs (no batch to pop, a first
// partial batch, no free slot, an output that ends early, an aborted heap)
// leaves everything as it is and plan->go at 0, and the per-batch kernel
// behind it does what there is to do.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "bgpq_device.hpp"
#include "bgpq_handle.hpp"

namespace bgpq {

namespace {

// A thread a key up to 1024: the walk is one workgroup's chain, and the merges
// are shorter with more threads.
constexpr int solo_threads(int B) { return B < 1024 ? B : 1024; }

template <typename K>
struct SoloArgs {
    K* items;
    int* ctr;
    K init_limits;
    int batch_num;
    int* go;
    const K* keys;  // inserted, `size` of them
    int size;
    K* out;
    long long out_cap;
};

template <typename K, bool BU, int B>
struct Solo {
    static constexpr int NT = solo_threads(B);
    static constexpr int kAhead = 4;  // levels of an insertion's path loaded ahead
    using Load = BatchLoad<K, B, NT>;
    static __device__ __forceinline__ int parent(int i) {
        if constexpr (BU) return (int)rev_idx(rev_idx((uint32_t)i) >> 1);
        else return i >> 1;
    }
    static __device__ __forceinline__ int child(int i, int right) {
        if constexpr (BU) return (int)rev_idx(rev_idx((uint32_t)i) << 1 | (uint32_t)right);
        else return i << 1 | right;
    }
    static __device__ __forceinline__ K* node(const SoloArgs<K>& a, int i) { return a.items + (size_t)i * B; }
    static __device__ __forceinline__ int& ctr(const SoloArgs<K>& a, int i) { return a.ctr[i * kWordStride]; }
    // Every wave's stores are acknowledged before any wave's loads after it.
    static __device__ __forceinline__ void publish() {
        wait_stores();
        __syncthreads();
    }

    static __device__ void insert(const SoloArgs<K>& a, K* X0, K* X1) {
        const int t = threadIdx.x, nb = ctr(a, CTR_BATCH_COUNT), pbs = ctr(a, CTR_PARTIAL);
        const bool whole = a.size + pbs >= B;  // a batch goes into the tree
        const bool ok = ctr(a, CTR_ABORT) == 0 && (whole ? nb < a.batch_num && (nb > 0 || a.size == B) : nb > 0);
        if (t == 0) *a.go = ok;
        if (!ok) return;
        if (!whole) {  // all keys to the partial buffer, by way of the root
            wg_sort_batch<K, B, NT>(X0, a.keys, a.size, a.init_limits);
            __syncthreads();
            g2l_batch<K, B, NT>(X1, node(a, 0));
            __syncthreads();
            wg_merge<K, B, NT>(X0, X1, ToLds<K>{X0}, ToNone{});
            g2l_batch<K, B, NT>(X1, node(a, 1));
            publish();
            wg_merge<K, B, NT>(X0, X1, ToGlobal<K>{node(a, 1)}, ToGlobal<K>{node(a, 0)});
            if (t == 0) ctr(a, CTR_PARTIAL) = pbs + a.size;
            return;
        }
        int cur = nb + 1, par = parent(cur), far = par;  // far: the next node to load
        Load path[kAhead];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            if (cur > 1 && far >= 1) {
                path[i].issue(node(a, far));
                far = far > 1 ? parent(far) : 0;
            }
        }
        wg_sort_batch<K, B, NT>(X0, a.keys, a.size, a.init_limits);
        __syncthreads();
        if (pbs > 0) {
            g2l_batch<K, B, NT>(X1, node(a, 0));
            publish();
            wg_merge<K, B, NT>(X0, X1, ToLds<K>{X0}, ToGlobal<K>{node(a, 0)});
        }
        bool done = cur == 1;
        while (!done) {
#pragma unroll
            for (int i = 0; i < kAhead; ++i) {
                if (!done) {
                    path[i].commit(X1);
                    if (far >= 1) {
                        path[i].issue(node(a, far));
                        far = far > 1 ? parent(far) : 0;
                    }
                    __syncthreads();
                    if (!(X0[0] < X1[B - 1])) {
                        done = true;  // the rest of the path is in order
                    } else {
                        wg_merge<K, B, NT>(X0, X1, ToLds<K>{X0}, ToGlobal<K>{node(a, cur)});
                        cur = par;
                        par = parent(par);
                        done = cur == 1;
                    }
                }
            }
        }
        l2g_batch<K, B, NT>(node(a, cur), X0);
        if (t == 0) {
            ctr(a, CTR_BATCH_COUNT) = nb + 1;
            ctr(a, CTR_PARTIAL) = pbs + a.size - B;
        }
    }

    static __device__ void remove(const SoloArgs<K>& a, K* X0, K* X1, K* X2) {
        const int t = threadIdx.x, nb = ctr(a, CTR_BATCH_COUNT), pbs = ctr(a, CTR_PARTIAL);
        const int off = ctr(a, CTR_DELETE_COUNT), last = nb;
        const bool ok = ctr(a, CTR_ABORT) == 0 && nb > 0 && off + (long long)B <= a.out_cap;
        if (t == 0) *a.go = ok;
        if (!ok) return;
        // the children, the last batch and the root at once
        Load l, r;
        int cl = 2, cr = 3;  // the children of node 1 in both orders
        if (cl < last) l.issue(node(a, cl));
        if (cr < last) r.issue(node(a, cr));
        if (last > 1) take_batch<K, B, NT>(X0, node(a, last), a.init_limits);
        K* const dst = a.out + off;
        if ((uintptr_t)dst % 16 == 0) {
            g2g_batch_last<K, B, NT>(dst, node(a, 1), key_slot<K>());
        } else {
            for (int i = t; i < B; i += NT) dst[i] = gload_key(node(a, 1) + i);
        }
        if (t == 0) {
            ctr(a, CTR_BATCH_COUNT) = nb - 1;
            ctr(a, CTR_DELETE_COUNT) = off + B;
            ctr(a, CTR_BUSY) += 1;  // the vote of a workgroup that popped
        }
        if (pbs > 0 && last > 1) {
            g2l_batch<K, B, NT>(X1, node(a, 0));
            publish();
            wg_merge<K, B, NT>(X0, X1, ToLds<K>{X0}, ToGlobal<K>{node(a, 0)});
        }
        if (last == 1) {
            publish();  // the root was read
            for (int i = t; i < B; i += NT) gstore_key(node(a, 1) + i, a.init_limits);
            return;
        }
        int cur = 1;
        for (;;) {
            // (a pop's first level also waits here for its reads of the root)
            if (cl < last) l.commit(X1);
            else fill_lds<K, B, NT>(X1, a.init_limits);
            if (cr < last) r.commit(X2);
            else fill_lds<K, B, NT>(X2, a.init_limits);
            if (cur == 1) wait_stores();
            __syncthreads();
            const K cmin = X0[0], cmax = X0[B - 1], kmin = X1[0] < X2[0] ? X1[0] : X2[0];
            if (!(kmin < cmax) || cl >= last) break;  // in order, or no child (cl < cr)
            // an absent child is the larger one, also beside keys that are not
            // below init_limits: the walk never leaves the slots in use
            const bool tr = cr >= last || X1[B - 1] < X2[B - 1];
            const int tgt = tr ? cr : cl, oth = tr ? cl : cr;
            cl = child(oth, 0);
            cr = child(oth, 1);
            if (cl < last) l.issue(node(a, cl));
            if (cr < last) r.issue(node(a, cr));
            if (tgt < last) wg_merge<K, B, NT>(X1, X2, ToLds<K>{X1}, ToGlobal<K>{node(a, tgt)});
            if (!(cmin < X1[B - 1])) l2g_batch<K, B, NT>(node(a, cur), X1);
            else wg_merge<K, B, NT>(X0, X1, ToGlobal<K>{node(a, cur)}, ToLds<K>{X0});
            __syncthreads();
            cur = oth;
        }
        l2g_batch<K, B, NT>(node(a, cur), X0);
    }
};

template <typename K, bool BU, int B, bool INSERT>
__global__ __launch_bounds__(solo_threads(B)) void k_solo(SoloArgs<K> a) {
    extern __shared__ __align__(16) int solo_lds[];
    K* const X = reinterpret_cast<K*>(solo_lds);
    if constexpr (INSERT) Solo<K, BU, B>::insert(a, X, X + B);
    else Solo<K, BU, B>::remove(a, X, X + B, X + 2 * B);
}

template <typename K, bool BU, int B, bool INSERT>
hipError_t launch(const SoloArgs<K>& a, hipEvent_t done, hipStream_t s) {
    constexpr int need = INSERT ? 2 * B * (int)sizeof(K) : 3 * B * (int)sizeof(K);
    constexpr int xch = INSERT ? sort_xch_bytes<K, B, solo_threads(B)>() : 0;
    constexpr int lds = need > xch ? need : xch;
    auto* const fn = &k_solo<K, BU, B, INSERT>;
    static const hipError_t ok =
        lds <= 64 * 1024 ? hipSuccess
                         : hipFuncSetAttribute(reinterpret_cast<const void*>(fn),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (ok != hipSuccess) return ok;
    clear_last_error();
    hipExtLaunchKernelGGL(fn, dim3(1), dim3(solo_threads(B)), lds, s, nullptr, done, 0, a);
    return hipGetLastError();
}

template <typename K, bool BU, bool INSERT>
hipError_t launch_b(const bgpq_heap* h, const SoloArgs<K>& a, hipStream_t s) {
    switch (h->batch_size) {
        case 64: return launch<K, BU, 64, INSERT>(a, h->bulk_done, s);
        case 128: return launch<K, BU, 128, INSERT>(a, h->bulk_done, s);
        case 256: return launch<K, BU, 256, INSERT>(a, h->bulk_done, s);
        case 512: return launch<K, BU, 512, INSERT>(a, h->bulk_done, s);
    }
    if constexpr (sizeof(K) == 4) {
        switch (h->batch_size) {
            case 1024: return launch<K, BU, 1024, INSERT>(a, h->bulk_done, s);
            case 2048: return launch<K, BU, 2048, INSERT>(a, h->bulk_done, s);
            case 4096: return launch<K, BU, 4096, INSERT>(a, h->bulk_done, s);
        }
    }
    return hipErrorInvalidValue;  // solo_pays refuses the others
}

template <typename K, bool INSERT>
hipError_t solo_as(const bgpq_heap* h, const void* keys, int size, void* out, long long out_cap, hipStream_t s) {
    const SoloArgs<K> a{(K*)h->items,       h->ctr,         (K)h->init_limits, h->batch_num, &h->bulk.plan->go,
                        (const K*)keys, size, (K*)out, out_cap};
    const bool bu = h->variant == BGPQ_BUITDD || h->variant == BGPQ_BUITDD_NP;
    return bu ? launch_b<K, true, INSERT>(h, a, s) : launch_b<K, false, INSERT>(h, a, s);
}

}  // namespace

bool solo_pays(const bgpq_heap* h) { return h->batch_size <= (h->key_type == BGPQ_KEY_U64 ? 512 : 4096); }
hipError_t solo_insert(const bgpq_heap* h, const void* keys, int size, hipStream_t s) {
    return h->key_type == BGPQ_KEY_U64 ? solo_as<uint64_t, true>(h, keys, size, nullptr, 0, s)
                                       : solo_as<uint32_t, true>(h, keys, size, nullptr, 0, s);
}
hipError_t solo_delete(const bgpq_heap* h, void* out, long long out_cap, hipStream_t s) {
    return h->key_type == BGPQ_KEY_U64 ? solo_as<uint64_t, false>(h, nullptr, 0, out, out_cap, s)
                                       : solo_as<uint32_t, false>(h, nullptr, 0, out, out_cap, s);
}

}  // namespace bgpq
