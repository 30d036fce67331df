// Kernels of the bulk insertion and deletion (bgpq_bulk.hpp) and their
// launch sequences.
//
//   k_plan_insert | k_plan_delete   what to do (BulkPlan), counters cleared
//   k_bulk_hist                     key counts of every digit of every pass
//   k_bulk_pass, once per digit     one pass of a least-digit-first radix sort
//   k_bulk_finish                   free slots refilled, counters set
//
// The passes follow the published single-pass scheme (decoupled look-back:
// Merrill and Garland, 2016; a radix pass on it: Adinets and Merrill, 2022):
// one read and one write of the keys per pass, where separate count and
// scatter kernels would read them twice.
#include <hip/hip_runtime.h>

#include "bgpq_device.hpp"
#include "bgpq_handle.hpp"

namespace bgpq {

namespace {

constexpr unsigned kLookCount = (1u << 30) - 1;  // lookback word: state << 30 | count
constexpr unsigned kLookOwn = 1u << 30;          // count of one tile
constexpr unsigned kLookAll = 2u << 30;          // count of the tile and all before it

__device__ __forceinline__ unsigned look_load(const unsigned* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void look_store(unsigned* p, unsigned v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename K>
__device__ __forceinline__ int digit_of(K k, int pass) {
    return (int)((k >> (8 * pass)) & (K)(kRadix - 1));
}

template <typename K>
__device__ __forceinline__ int ctr_of(const BulkArgs<K>& a, int i) {
    return a.ctr[i * kWordStride];
}

// Key j of the heap's keys (partial buffer, then slots 1, 2, ...) and the
// new ones after them: the order the sort reads them in.
template <typename K>
__device__ __forceinline__ const K* source_key(const BulkArgs<K>& a, const BulkPlan& pl, int j) {
    const int held = pl.pbs + pl.nb * a.batch_size;
    if (j >= held) return a.keys + (j - held);
    return j < pl.pbs ? a.items + j : a.items + a.batch_size + (j - pl.pbs);
}

// Address of key 0 such that keys j .. j + len - 1 follow each other from
// there, or null where they cross from one part to the next.
template <typename K>
__device__ __forceinline__ const K* source_run(const BulkArgs<K>& a, const BulkPlan& pl, int j, int len) {
    const int held = pl.pbs + pl.nb * a.batch_size;
    if (j + len > pl.total) return nullptr;
    if (j >= held) return a.keys - held;
    return j >= pl.pbs && j + len <= held ? a.items + (a.batch_size - pl.pbs) : nullptr;
}

// Where sorted key j goes: the output first, then slots 1, 2, ... of the
// heap, the largest into the partial buffer.
template <typename K>
__device__ __forceinline__ K* final_place(const BulkArgs<K>& a, const BulkPlan& pl, int j) {
    if (j < pl.cut) return a.out + pl.off + j;
    j -= pl.cut;
    return j < pl.full_after ? a.items + a.batch_size + j : a.items + (j - pl.full_after);
}

// Counters of the sort back to zero (one workgroup).
__device__ __forceinline__ void clear_sort_words(const BulkMem& m) {
    for (int i = threadIdx.x; i < kMaxPasses * kRadix; i += blockDim.x) m.hist[i] = 0;
    if (threadIdx.x < kMaxPasses) m.ticket[threadIdx.x] = 0;
}

// The workgroup that arrives last at a grid-wide counter: it sees what the
// others added before they arrived (device-scope atomics and loads only).
__device__ __forceinline__ bool last_to_arrive(int* arrived) {
    __shared__ int s_last;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) s_last = a_add(arrived, 1) == (int)gridDim.x - 1;
    __syncthreads();
    return s_last != 0;
}

// The plan's part that a call's pops decide: a.calls of them from nb batches
// and pbs partial keys, whole batches first and the partial buffer only once
// no batch is left, as many as the output holds.  The slots in use end below
// `spare`; `through` keys pass through the free slots from there on.
template <typename K>
__device__ __forceinline__ void plan_pops(const BulkArgs<K>& a, BulkPlan& pl, long long nb, int pbs, long long spare,
                                          bool ascending) {
    const long long B = a.batch_size, total = nb * B + pbs, off = ctr_of(a, CTR_DELETE_COUNT);
    long long pops = a.calls < nb ? a.calls : nb;
    const long long room = off <= a.out_cap ? (a.out_cap - off) / B : 0;
    int error = 0;
    if (pops > room) {
        pops = room;
        error = ERR_OUTPUT_FULL;
    }
    bool last = pops == nb && a.calls > nb && pbs > 0;
    if (last && off + total > a.out_cap) {
        last = false;
        error = ERR_OUTPUT_FULL;
    }
    const long long cut = pops * B + (last ? pbs : 0);
    const long long tiles = (total + bulk_tile<K>() - 1) / bulk_tile<K>();
    pl.total = (int)total;
    pl.tiles = (int)tiles;
    pl.ascending = ascending;
    pl.cut = (int)cut;
    pl.off = (int)off;
    pl.nb_after = (int)(nb - pops);
    pl.pbs_after = last ? 0 : pbs;
    pl.full_after = (int)((nb - pops) * B);
    // a sort moves every key through the free slots, ascending slots only
    // the batches that stay (the partial buffer stays where it is)
    const long long through = ascending ? (nb - pops) * B : total;
    pl.spare = spare;
    pl.fill_lo = (nb - pops + 1) * B;
    pl.fill_hi = spare + through;
    pl.error = error;
    pl.idle = a.calls > pops + (last ? 1 : 0) && total == cut;
    pl.go = total > 0 && total < kBulkMaxKeys && tiles <= a.mem.tiles_max &&
            spare + through <= ((long long)a.batch_num + 1) * B && (cut == 0 || off + total < (1ll << 31)) &&
            ctr_of(a, CTR_ABORT) == 0;
}

// Insertions, and pops after them where the call has any (a concurrent call,
// whose insertions and pops may take effect in any order).
template <typename K>
__global__ __launch_bounds__(256) void k_plan_insert(BulkArgs<K> a) {
    BulkPlan& pl = *a.mem.plan;
    clear_sort_words(a.mem);
    if (threadIdx.x != 0) return;
    const int B = a.batch_size, nb = ctr_of(a, CTR_BATCH_COUNT), pbs = ctr_of(a, CTR_PARTIAL);
    const long long total = (long long)nb * B + pbs + a.n, full = total / B;
    pl.nb = nb;
    pl.pbs = pbs;
    plan_pops(a, pl, full, (int)(total % B), (full + 1) * B, false);
    if (full > a.batch_num) pl.go = 0;
}

// Pops alone.  Do the slots ascend already (a bulk insertion leaves them so)?
// Each batch ascends by itself, so only the borders are compared.
template <typename K>
__global__ __launch_bounds__(256) void k_plan_delete(BulkArgs<K> a) {
    BulkPlan& pl = *a.mem.plan;
    const int B = a.batch_size, nb = ctr_of(a, CTR_BATCH_COUNT), pbs = ctr_of(a, CTR_PARTIAL);
    bool bad = false;
    for (long long i = blockIdx.x * 256ll + threadIdx.x; i < nb; i += gridDim.x * 256ll) {
        const K end = a.items[(i + 2) * B - 1];
        if (i + 1 < nb) bad |= a.items[(i + 2) * B] < end;
        else if (pbs > 0) bad |= a.items[0] < end;
    }
    if (__any(bad) && __lane_id() == 0) a_add(&pl.violations, 1);
    if (!last_to_arrive(&pl.arrived)) return;
    clear_sort_words(a.mem);
    if (threadIdx.x != 0) return;
    const bool ascending = a_load(&pl.violations) == 0;
    a_store(&pl.violations, 0);
    a_store(&pl.arrived, 0);
    pl.nb = nb;
    pl.pbs = pbs;
    plan_pops(a, pl, nb, pbs, (nb + 1ll) * B, ascending);
    if (pl.cut == 0) pl.go = 0;  // nothing to do but what the per-batch kernel reports
}

// Key counts of each digit.  A wave whose keys agree on a digit (ordered or
// small keys: the high digits) adds its 64 at once instead of serialising on
// one word.  The last workgroup turns the counts into first positions and
// drops the passes whose digit is the same for all keys; the number of
// passes left is made even, so that the sort ends where it began.
template <typename K>
__global__ __launch_bounds__(256) void k_bulk_hist(BulkArgs<K> a) {
    constexpr int P = (int)sizeof(K), U = 16;
    __shared__ unsigned h[P][kRadix];
    __shared__ unsigned part[4];
    __shared__ int moves[P];
    BulkPlan& pl = *a.mem.plan;
    if (!pl.go || pl.ascending) return;
    const int t = threadIdx.x, total = pl.total;
    for (int i = t; i < P * kRadix; i += 256) (&h[0][0])[i] = 0;
    __syncthreads();
    // the first pass's lookback words
    for (long long i = blockIdx.x * 256ll + t; i < (long long)pl.tiles * kRadix; i += gridDim.x * 256ll)
        a.mem.look[0][i] = 0;
    for (long long j0 = (long long)blockIdx.x * (256 * U); j0 < total; j0 += (long long)gridDim.x * (256 * U)) {
        K k[U];
        const int j = (int)j0 + t;
        if (const K* src = source_run(a, pl, (int)j0, 256 * U)) {
#pragma unroll
            for (int u = 0; u < U; ++u) k[u] = src[j + u * 256];
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u) k[u] = j + u * 256 < total ? *source_key(a, pl, j + u * 256) : K(0);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool in = j + u * 256 < total;
            const bool whole = __ballot(in) == ~0ull;
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const int d = digit_of(k[u], p);
                const int d0 = __builtin_amdgcn_readfirstlane(d);
                if (whole && __ballot(d == d0) == ~0ull) {
                    if (__lane_id() == 0) atomicAdd(&h[p][d0], 64u);
                } else if (in) {
                    atomicAdd(&h[p][d], 1u);
                }
            }
        }
    }
    __syncthreads();
    for (int i = t; i < P * kRadix; i += 256) {
        const unsigned c = (&h[0][0])[i];
        if (c) __hip_atomic_fetch_add(a.mem.hist + i, c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (!last_to_arrive(&pl.arrived)) return;
    const int lane = t & 63, w = t >> 6;
    for (int p = 0; p < P; ++p) {
        const unsigned c = look_load(a.mem.hist + p * kRadix + t);
        unsigned x = c;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (lane == 63) part[w] = x;
        if (t == 0) moves[p] = 1;
        __syncthreads();
        if (c == (unsigned)total) moves[p] = 0;
        unsigned before = 0;
        for (int i = 0; i < w; ++i) before += part[i];
        a.mem.hist[p * kRadix + t] = x - c + before;
        __syncthreads();
    }
    if (t == 0) {
        int n = 0;
        for (int p = 0; p < P; ++p) n += moves[p];
        for (int p = 0; p < P && (n < 2 || (n & 1)); ++p) {
            if (!moves[p]) {
                moves[p] = 1;
                ++n;
            }
        }
        int at = 0;
        for (int p = 0; p < P; ++p) pl.order[p] = moves[p] ? at++ : -1;
        pl.active = n;
        a_store(&pl.arrived, 0);
    }
}

// The slots already ascend: keys to be handed out go to the output, batches
// that stay to the spare slots (k_bulk_finish brings them back).
template <typename K>
__device__ void copy_ascending(const BulkArgs<K>& a, const BulkPlan& pl) {
    constexpr int U = 8;
    const int full = pl.nb * a.batch_size, moved = pl.cut + pl.full_after;
    const long long step = (long long)gridDim.x * kBulkThreads * U;
    for (long long j0 = (long long)blockIdx.x * (kBulkThreads * U); j0 < moved; j0 += step) {
        const int j = (int)j0 + (int)threadIdx.x;
        K k[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = j + u * kBulkThreads;
            if (i < moved) k[u] = i < full ? a.items[a.batch_size + i] : a.items[i - full];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = j + u * kBulkThreads;
            if (i < moved) *(i < pl.cut ? a.out + pl.off + i : a.items + pl.spare + (i - pl.cut)) = k[u];
        }
    }
}

// One pass: the keys, in their present order, to the places their digit's
// counts give.  Workgroups take tiles by ticket, so every tile before theirs
// is finished or running and the look-back ends.
//   * Each wave ranks its keys by digit with ballots (64 keys at a time, in
//     order, so the pass is stable), counting in a table of its own.
//   * 256 threads, one per digit, publish the tile's counts and look back
//     for those of the tiles before it; meanwhile the keys move into LDS in
//     digit order, from where each digit's run is written as a whole.
template <typename K>
__global__ __launch_bounds__(kBulkThreads, 4) void k_bulk_pass(BulkArgs<K> a, int pass) {
    constexpr int T = bulk_tile<K>(), U = T / kBulkThreads, W = kBulkThreads / 64;
    __shared__ K keys[T];
    __shared__ unsigned cnt[W][kRadix];
    __shared__ unsigned to[kRadix];
    __shared__ unsigned part[4];
    __shared__ int s_tile;
    const BulkPlan& pl = *a.mem.plan;
    if (!pl.go) return;
    if (pl.ascending) {
        if (pass == 0) copy_ascending(a, pl);
        return;
    }
    const int ord = pl.order[pass];
    if (ord < 0) return;
    const bool first = ord == 0, last = ord == pl.active - 1;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int total = pl.total, tiles = pl.tiles;
    K* const spare = a.items + pl.spare;
    const K* const src = (ord & 1) ? spare : a.items;
    K* const dst = (ord & 1) ? a.items : spare;
    unsigned* const look = a.mem.look[ord & 1];
    unsigned* const next = last ? nullptr : a.mem.look[(ord & 1) ^ 1];
    const unsigned start = t < kRadix ? a.mem.hist[pass * kRadix + t] : 0;
    const unsigned long long below = (1ull << lane) - 1;
    for (;;) {
        if (t == 0) s_tile = (int)atomicAdd(a.mem.ticket + pass, 1u);
#pragma unroll
        for (int i = 0; i < W * kRadix / kBulkThreads; ++i) (&cnt[0][0])[i * kBulkThreads + t] = 0;
        __syncthreads();
        const int tile = s_tile;
        if (tile >= tiles) break;
        const int j0 = tile * T, j = j0 + w * (64 * U) + lane;
        const int here = total - j0 < T ? total - j0 : T;
        K k[U];
        const K* const run = first ? source_run(a, pl, j0, T) : (here == T ? src : nullptr);
        if (run) {
#pragma unroll
            for (int u = 0; u < U; ++u) k[u] = run[j + u * 64];
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = j + u * 64;
                k[u] = i < total ? (first ? *source_key(a, pl, i) : src[i]) : ~K(0);
            }
        }
        // ranks among the wave's keys of the same digit (keys past the end
        // count as digit 255 and come last)
        unsigned short rank[U];
        unsigned* const mine = cnt[w];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int d = digit_of(k[u], pass);
            unsigned long long same = ~0ull;
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const bool bit = (d >> b) & 1;
                const unsigned long long m = __ballot(bit);
                same &= bit ? m : ~m;
            }
            const unsigned before = mine[d];
            const int ahead = __popcll(same & below);
            rank[u] = (unsigned short)(before + ahead);
            __builtin_amdgcn_wave_barrier();
            if (ahead == 0) mine[d] = before + __popcll(same);
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
        unsigned own = 0, upto = 0, of_wave[W];
        if (t < kRadix) {
#pragma unroll
            for (int i = 0; i < W; ++i) {
                of_wave[i] = own;
                own += cnt[i][t];
            }
            upto = own;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const unsigned y = __shfl_up(upto, o, 64);
                if (lane >= o) upto += y;
            }
            if (lane == 63) part[w] = upto;
            upto -= own;
            if (t == kRadix - 1) own -= T - here;  // padding does not count
            look_store(look + (size_t)tile * kRadix + t, (tile == 0 ? kLookAll : kLookOwn) | own);
            if (next) next[(size_t)tile * kRadix + t] = 0;
        }
        __syncthreads();
        if (t < kRadix) {
            for (int i = 0; i < w; ++i) upto += part[i];  // first place of the digit in the tile
#pragma unroll
            for (int i = 0; i < W; ++i) cnt[i][t] = upto + of_wave[i];
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < U; ++u) keys[mine[digit_of(k[u], pass)] + rank[u]] = k[u];
        unsigned before = 0;
        if (t < kRadix && tile > 0) {
            const unsigned* p = look + (size_t)(tile - 1) * kRadix + t;
            int polls = 0;
            for (int back = tile - 1;;) {
                const unsigned v = look_load(p);
                if ((v >> 30) == 0) {
                    // the tile before is running; the bound only ends a fault
                    if (++polls > kSpinLimit) {
                        __hip_atomic_fetch_or(a.ctr + CTR_ERROR * kWordStride, (int)ERR_SPIN_LIMIT, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT);
                        break;
                    }
                    continue;
                }
                before += v & kLookCount;
                if ((v >> 30) == 2 || back == 0) break;
                --back;
                p -= kRadix;
            }
            look_store(look + (size_t)tile * kRadix + t, kLookAll | (before + own));
        }
        if (t < kRadix) to[t] = start + before - upto;  // place of a key = to[digit] + its place in the tile
        __syncthreads();
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = u * kBulkThreads + t;
            if (i < here) {
                const K key = keys[i];
                const int at = (int)to[digit_of(key, pass)] + i;
                if (last) *final_place(a, pl, at) = key;
                else dst[at] = key;
            }
        }
    }
}

// Batches that stay come back from the spare slots (ascending slots only);
// the slots that are free now hold init_limits again; the counters follow.
template <typename K>
__global__ __launch_bounds__(256) void k_bulk_finish(BulkArgs<K> a) {
    const BulkPlan& pl = *a.mem.plan;
    if (!pl.go) return;
    const long long i0 = blockIdx.x * 256ll + threadIdx.x, step = gridDim.x * 256ll;
    const K v = a.init_limits;
    long long lo = pl.fill_lo;
    const long long hi = pl.fill_hi;
    if (pl.ascending && pl.full_after > 0) {
        K* const spare = a.items + pl.spare;
        for (long long i = i0; i < pl.full_after; i += step) {
            a.items[a.batch_size + i] = spare[i];
            spare[i] = v;
        }
        for (long long i = lo + i0; i < pl.spare; i += step) a.items[i] = v;
    } else {
        constexpr int V = 16 / (int)sizeof(K);
        typedef K vec __attribute__((ext_vector_type(V)));
        vec q;
#pragma unroll
        for (int i = 0; i < V; ++i) q[i] = v;
        // lo is a multiple of the batch size
        for (long long i = lo / V + i0; i < hi / V; i += step) reinterpret_cast<vec*>(a.items)[i] = q;
        if (i0 < hi % V) a.items[hi / V * V + i0] = v;
    }
    if (!(pl.ascending && pl.pbs_after == pl.pbs))
        for (long long i = pl.pbs_after + i0; i < a.batch_size; i += step) a.items[i] = v;
    if (i0 == 0) {
        a.ctr[CTR_BATCH_COUNT * kWordStride] = pl.nb_after;
        a.ctr[CTR_PARTIAL * kWordStride] = pl.pbs_after;
        a.ctr[CTR_DELETE_COUNT * kWordStride] += pl.cut;
        a.ctr[CTR_ERROR * kWordStride] |= pl.error;
        if (pl.idle && a.ctr[CTR_BUSY * kWordStride] <= 0) a.ctr[CTR_TERM * kWordStride] = 1;
    }
}

inline int blocks_for(long long items, int per_block, int most) {
    const long long b = (items + per_block - 1) / per_block;
    return (int)(b < 1 ? 1 : (b > most ? most : b));
}

template <typename K>
hipError_t sort_and_finish(const BulkArgs<K>& a, long long keys, int cus, hipStream_t s) {
    hipLaunchKernelGGL(k_bulk_hist<K>, dim3(blocks_for(keys, 4096, 4 * cus)), dim3(256), 0, s, a);
    const int grid = blocks_for(keys, bulk_tile<K>(), 3 * cus);
    for (int p = 0; p < (int)sizeof(K); ++p)
        hipLaunchKernelGGL(k_bulk_pass<K>, dim3(grid), dim3(kBulkThreads), 0, s, a, p);
    hipLaunchKernelGGL(k_bulk_finish<K>, dim3(blocks_for(keys, 4096, 8 * cus)), dim3(256), 0, s, a);
    return hipGetLastError();
}

template <typename K>
BulkArgs<K> args_for(const bgpq_heap* h) {
    BulkArgs<K> a{};
    a.items = (K*)h->items;
    a.ctr = h->ctr;
    a.init_limits = (K)h->init_limits;
    a.batch_num = h->batch_num;
    a.batch_size = h->batch_size;
    a.mem = h->bulk;
    return a;
}

template <typename K>
hipError_t insert_as(const bgpq_heap* h, const void* keys, long long n, void* out, long long out_cap, long long calls,
                     int cus, hipStream_t s) {
    BulkArgs<K> a = args_for<K>(h);
    a.keys = (const K*)keys;
    a.n = n;
    a.out = (K*)out;
    a.out_cap = out_cap;
    a.calls = calls;
    clear_last_error();
    hipLaunchKernelGGL(k_plan_insert<K>, dim3(1), dim3(256), 0, s, a);
    return sort_and_finish(a, h->held + n, cus, s);
}

template <typename K>
hipError_t delete_as(const bgpq_heap* h, void* out, long long out_cap, long long calls, int cus, hipStream_t s) {
    BulkArgs<K> a = args_for<K>(h);
    a.out = (K*)out;
    a.out_cap = out_cap;
    a.calls = calls;
    clear_last_error();
    hipLaunchKernelGGL(k_plan_delete<K>, dim3(blocks_for(h->held / h->batch_size, 256, cus)), dim3(256), 0, s, a);
    return sort_and_finish(a, h->held, cus, s);
}

}  // namespace

hipError_t bulk_insert(const bgpq_heap* h, const void* keys, long long n, void* out, long long out_cap,
                       long long calls, int cus, hipStream_t s) {
    return h->key_type == BGPQ_KEY_U64 ? insert_as<uint64_t>(h, keys, n, out, out_cap, calls, cus, s)
                                       : insert_as<uint32_t>(h, keys, n, out, out_cap, calls, cus, s);
}
hipError_t bulk_delete(const bgpq_heap* h, void* out, long long out_cap, long long calls, int cus, hipStream_t s) {
    return h->key_type == BGPQ_KEY_U64 ? delete_as<uint64_t>(h, out, out_cap, calls, cus, s)
                                       : delete_as<uint32_t>(h, out, out_cap, calls, cus, s);
}

}  // namespace bgpq
