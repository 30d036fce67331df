// Kernels of the bulk insertion and deletion (bgpq_bulk.hpp) and their
// launch sequences.
//
// A sort (insertions, pops from slots in heap order):
//   k_plan_delete                   pops only: what to do (BulkPlan)
//   k_bulk_hist                     key counts of every digit of every pass
//                                   (and the plan, where there are insertions)
//   k_bulk_pass, a launch a digit   one pass of a least-digit-first radix sort
//   k_bulk_finish                   free slots refilled, counters set
// or, for insertions that make no more than a tile of keys in all, with pops or
// without, k_bulk_tile alone.
// Pops from slots that ascend, as a bulk call leaves them:
//   k_plan_delete, k_bulk_copy, k_bulk_finish
//
// The passes follow the published single-pass scheme (decoupled look-back:
// Merrill and Garland, 2016; a radix pass on it: Adinets and Merrill, 2022):
// one read and one write of the keys per pass, where separate count and
// scatter kernels would read them twice.
#include <hip/hip_ext.h>
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

// The loop behind it starts on a line of the instruction cache, in a pass of the
// large tiles.  Its loops are long and run from there again and again: where
// they happened to start made up to 2% of a sort (12.3 M descending u32 keys 276.5
// and 283 us with the same instructions 16 bytes apart, 279 aligned; 2^28 random
// 3197, 3207, 3174).  In a pass of the small tiles it gained nothing (rounds of
// 1.5 M u64 keys in all 971 us, 967 without).
template <typename K, int T>
__device__ __forceinline__ void align_loop() {
    if constexpr (T == bulk_tile<K>(true)) asm volatile(".p2align 6");
}

// The same value as one the compiler knows nothing of: what is computed from
// it is computed anew, not kept in registers from the last use on.
__device__ __forceinline__ int anew(int x) {
    asm volatile("" : "+s"(x));
    return x;
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
    // a call without pops has nothing to do with the cursor, which the host may
    // set at any time (bgpq_set_cursor is not ordered on the heap's stream)
    const long long B = a.batch_size, total = nb * B + pbs;
    const long long off = a.from_empty || a.calls == 0 ? 0 : ctr_of(a, CTR_DELETE_COUNT);
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
    const long long tiles = (total + a.tile - 1) / a.tile;
    pl.total = (int)total;
    pl.tiles = (int)tiles;
    pl.ascending = ascending;
    pl.drains = total == cut;
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
    // The vote as the workgroups of a per-batch call would leave it, each with
    // every `poppers`th call, the calls in order: a workgroup is busy from its
    // first pop until a call of its finds nothing, and those calls come last.
    const long long none = a.calls - pops - (last ? 1 : 0);
    const long long workgroups = a.calls < a.poppers ? a.calls : a.poppers;
    pl.idle = none > 0;
    pl.busy = (int)(workgroups - (none < workgroups ? none : workgroups));
    pl.go = total > 0 && total < kBulkMaxKeys && tiles <= a.mem.tiles_max &&
            spare + through <= ((long long)a.batch_num + 1) * B && (cut == 0 || off + total < (1ll << 31)) &&
            ctr_of(a, CTR_ABORT) == 0;
}

// Insertions, and pops after them where the call has any (a concurrent call,
// whose insertions and pops may take effect in any order, or a heap sort).
template <typename K>
__device__ __forceinline__ void plan_insert(const BulkArgs<K>& a, BulkPlan& pl) {
    const int B = a.batch_size, nb = ctr_of(a, CTR_BATCH_COUNT), pbs = ctr_of(a, CTR_PARTIAL);
    const long long total = (long long)nb * B + pbs + a.n, full = total / B;
    pl.nb = nb;
    pl.pbs = pbs;
    plan_pops(a, pl, full, (int)(total % B), (full + 1) * B, false);
    if (full > a.batch_num || (a.from_empty && (nb | pbs) != 0)) pl.go = 0;
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
    if (__any(bad) && __lane_id() == 0) a_add(a.mem.sync, 1);
    if (!last_to_arrive(a.mem.sync + 1)) return;
    if (threadIdx.x != 0) return;
    const bool ascending = a_load(a.mem.sync) == 0;
    a_store(a.mem.sync, 0);
    a_store(a.mem.sync + 1, 0);
    pl.nb = nb;
    pl.pbs = pbs;
    plan_pops(a, pl, nb, pbs, (nb + 1ll) * B, ascending);
    // nothing to do but what the per-batch kernel reports, or a sort that was not launched
    if (pl.cut == 0 || !(ascending || a.sorts)) pl.go = 0;
}

// Key counts of each digit: LDS atomics, of which a wave whose keys agree on
// a digit (ordered or small keys: the high digits) makes one instead of 64 on
// one word.  The rows of 64 keys are looked at one by one only where the first
// agrees; a test of every row cost as much as the atomics.  The last
// workgroup turns the counts into first positions and drops the passes whose
// digit is the same for all keys.  The first pass must not write where keys
// are read, so at least two are left; an even number, so that the sort ends
// where it began, unless the last pass hands every key out.
template <typename K>
__global__ __launch_bounds__(256) void k_bulk_hist(BulkArgs<K> a) {
    constexpr int P = (int)sizeof(K), U = 16;
    __shared__ unsigned h[P][kRadix];
    __shared__ int moves[P];
    __shared__ BulkPlan pl;
    const int t = threadIdx.x;
    if (t == 0) {
        if (a.planned) pl = *a.mem.plan;
        else plan_insert(a, pl);
        if (!pl.go && blockIdx.x == 0) a.mem.plan->go = 0;
    }
    for (int i = t; i < P * kRadix; i += 256) (&h[0][0])[i] = 0;
    __syncthreads();
    if (!pl.go || pl.ascending) return;
    const int total = pl.total;
    // the first pass's lookback words
    for (long long i = blockIdx.x * 256ll + t; i < (long long)pl.tiles * kRadix; i += gridDim.x * 256ll)
        a.mem.look[0][i] = 0;
    for (long long j0 = (long long)blockIdx.x * (256 * U); j0 < total; j0 += (long long)gridDim.x * (256 * U)) {
        K k[U];
        const int j = (int)j0 + t;
        if (const K* src = source_run(a, pl, (int)j0, 256 * U)) {
#pragma unroll
            for (int u = 0; u < U; ++u) k[u] = src[j + u * 256];
#pragma unroll
            for (int p = 0; p < P; ++p) {
                if (__ballot(digit_of(k[0], p) == __builtin_amdgcn_readfirstlane(digit_of(k[0], p))) != ~0ull) {
#pragma unroll
                    for (int u = 0; u < U; ++u) atomicAdd(&h[p][digit_of(k[u], p)], 1u);
                } else {
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int d = digit_of(k[u], p), d0 = __builtin_amdgcn_readfirstlane(d);
                        if (__ballot(d == d0) != ~0ull) atomicAdd(&h[p][d], 1u);
                        else if (__lane_id() == 0) atomicAdd(&h[p][d0], 64u);
                    }
                }
            }
        } else {
            for (int u = 0; u < U && j + u * 256 < total; ++u) {
                const K key = *source_key(a, pl, j + u * 256);
#pragma unroll
                for (int p = 0; p < P; ++p) atomicAdd(&h[p][digit_of(key, p)], 1u);
            }
        }
    }
    __syncthreads();
    for (int i = t; i < P * kRadix; i += 256) {
        const unsigned c = (&h[0][0])[i];
        if (c) __hip_atomic_fetch_add(a.mem.hist + i, c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (!last_to_arrive(a.mem.sync + 1)) return;
    // a wave for every fourth digit, four counts a lane (a barrier for each
    // digit's scan took 2 of the kernel's 20 us for 250,000 u64 keys)
    const int lane = t & 63;
#pragma unroll
    for (int p = t >> 6; p < P; p += 4) {
        unsigned* const at = a.mem.hist + p * kRadix + lane * 4;
        unsigned c[4], sum = 0;
        bool same = false;
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i] = look_load(at + i);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            same |= c[i] == (unsigned)total;
            sum += c[i];
        }
        unsigned x = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        x -= sum;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            at[i] = x;
            x += c[i];
        }
        const bool any = __any(same);
        if (lane == 0) moves[p] = !any;
    }
    __syncthreads();
    if (t == 0) {
        int n = 0;
        for (int p = 0; p < P; ++p) n += moves[p];
        for (int p = 0; p < P && (n < 2 || ((n & 1) && !pl.drains)); ++p) {
            if (!moves[p]) {
                moves[p] = 1;
                ++n;
            }
        }
        // dropped passes are the first launches: the last one always hands the keys out
        int at = 0;
        for (int p = 0; p < P - n; ++p) pl.order[p] = -1;
        for (int p = 0; p < P; ++p) {
            if (moves[p]) {
                pl.order[P - n + at] = at << 8 | p;
                ++at;
            }
        }
        pl.active = n;
        // where all keys leave, the output is the second buffer, so that the
        // slots in use need no refill twice as long as the keys
        pl.through_out = pl.drains && (n & 1) == 0;
        if (pl.through_out && pl.nb == 0 && pl.pbs == 0) pl.fill_lo = pl.spare;
        *a.mem.plan = pl;
        a_store(a.mem.sync + 1, 0);
    }
}

// The slots already ascend: keys to be handed out go to the output, batches
// that stay to the spare slots (k_bulk_finish brings them back).
template <typename K>
__global__ __launch_bounds__(kBulkThreads) void k_bulk_copy(BulkArgs<K> a) {
    constexpr int U = 8;
    const BulkPlan& pl = *a.mem.plan;
    if (!pl.go || !pl.ascending) return;
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

template <int H>
__device__ __forceinline__ unsigned rank_of(const unsigned (&rank)[H], int u) {
    return u % 2 == 0 ? rank[u / 2] & 0xFFFFu : rank[u / 2] >> 16;
}
// Ranks of the wave's keys, U rows of 64, among those of the same digit, in
// order, and the digits' counts in `mine` (zeroed before): most of a pass's
// vector instructions, and 3 LDS accesses a row.  A lane finds the lanes with its
// digit bit by bit: one ballot and one v_bitop3 for each half of the mask.
// The ranks are kept two to a register: with 32 rows' keys and ranks in
// registers of their own the large tiles of u32 keys spilled, which wrote 1.7
// bytes for each byte sorted (790 us a pass at 2^28 keys, 700 so).
template <typename K, int U>
__device__ __forceinline__ void rank_rows(const K (&k)[U], int pass, unsigned* mine, unsigned (&rank)[U / 2]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int d = digit_of(k[u], pass);
        unsigned lo = ~0u, hi = ~0u;  // lanes with the same digit
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            int bit = __builtin_amdgcn_sbfe(d, b, 1);
            asm("" : "+v"(bit));  // compared as it is, not shifted anew
            const unsigned long long m = __ballot(bit != 0);
            lo = __builtin_amdgcn_bitop3_b32(lo, (unsigned)m, (unsigned)bit, 0x90);  // lo & ~(m ^ bit)
            hi = __builtin_amdgcn_bitop3_b32(hi, (unsigned)(m >> 32), (unsigned)bit, 0x90);
        }
        const unsigned ahead = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0));
        const unsigned both = ahead | (unsigned)(__popc(lo) + __popc(hi)) << 8;
        rank[u / 2] = u % 2 == 0 ? both : rank[u / 2] | both << 16;
        // one row's masks at a time, and the test for a digit's first lane
        // not before it is needed: 16 rows' masks would spill
        asm volatile("" : "+v"(rank[u / 2]));
        __builtin_amdgcn_sched_barrier(0);
    }
    const int again = anew(pass);
#pragma unroll
    for (int u = 0; u < U; ++u) {
        unsigned* const c = mine + digit_of(k[u], again);
        const unsigned before = *c, both = rank_of(rank, u), ahead = both & 0xFFu;
        __builtin_amdgcn_wave_barrier();
        if (ahead == 0) *c = before + (both >> 8);
        __builtin_amdgcn_wave_barrier();
        const unsigned r = before + ahead;  // below 2^16, like both
        rank[u / 2] = u % 2 == 0 ? (rank[u / 2] & 0xFFFF0000u) | r : (rank[u / 2] & 0xFFFFu) | r << 16;
    }
}

// Thread t < 256: digit t's count in the tile (own), its keys' places before
// each wave's (of_wave), and the sum of the lower digits' counts in t's wave
// (upto) and, for all, in part[].
template <int W>
__device__ __forceinline__ void count_digits(const unsigned (&cnt)[W][kRadix], unsigned* part, unsigned& own,
                                             unsigned& upto, unsigned (&of_wave)[W]) {
    const int t = threadIdx.x, lane = t & 63;
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
    if (lane == 63) part[t >> 6] = upto;
    upto -= own;
}

// One pass: the keys, in their present order, to the places their digit's
// counts give.  Workgroups take tiles by ticket, so every tile before theirs
// is finished or running and the look-back ends.
//   * Each wave ranks its keys by digit with ballots (64 keys at a time, in
//     order, so the pass is stable), counting in a table of its own.
//   * 256 threads, one per digit, publish the tile's counts and look back
//     for those of the tiles before it; meanwhile the keys move into LDS in
//     digit order, from where each digit's run is written as a whole.
// What bounds it: vector instructions (69 for 64 keys, 75% of the cycles at 2^28
// u32 keys) and waits for LDS and memory; 694 us a pass there, 3.1 TB/s read
// and written where a copy reaches 4.6.  It took 1150 us with lane masks built
// by selects (95 instructions for the ranks alone; a mask's step is one
// v_bitop3 now) and a look-back of one tile at a time, each a round trip of
// about a microsecond.
template <typename K, int T>
__global__ __launch_bounds__(kBulkThreads, 4) void k_bulk_pass(BulkArgs<K> a, int launch) {
    constexpr int U = T / kBulkThreads, W = kBulkThreads / 64;
    constexpr int kWindow = 16;  // tiles looked at together
    __shared__ K keys[T];
    __shared__ unsigned cnt[W][kRadix];
    __shared__ unsigned to[kRadix];
    __shared__ unsigned part[4];
    __shared__ int s_tile;
    const BulkPlan& pl = *a.mem.plan;
    if (!pl.go || pl.ascending) return;
    const int order = pl.order[launch];
    if (order < 0) return;
    const int ord = order >> 8, pass = order & 0xFF;
    const bool first = ord == 0, last = ord == pl.active - 1;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int total = pl.total, tiles = pl.tiles;
    K* const spare = a.items + pl.spare;
    K* const second = pl.through_out ? a.out + pl.off : a.items;
    const K* const src = (ord & 1) ? spare : second;
    // the last pass's places are not in a row where some keys stay
    const bool split = last && !pl.drains;
    K* const dst = last ? a.out + pl.off : (ord & 1) ? second : spare;
    unsigned* const look = a.mem.look[ord & 1];
    unsigned* const next = last ? nullptr : a.mem.look[(ord & 1) ^ 1];
    const unsigned start = t < kRadix ? a.mem.hist[pass * kRadix + t] : 0;
    align_loop<K, T>();
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
            // the last tile, and those across two parts of the source
#pragma unroll 1
            for (int u = 0; u < U; ++u) {
                const int i = j + u * 64;
                keys[i - j0] = i < total ? *(first ? source_key(a, pl, i) : src + i) : ~K(0);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) k[u] = keys[j - j0 + u * 64];  // a thread reads back its own
        }
        unsigned rank[U / 2];
        unsigned* const mine = cnt[w];
        rank_rows(k, pass, mine, rank);
        __syncthreads();
        unsigned own = 0, upto = 0, of_wave[W];
        if (t < kRadix) {
            count_digits(cnt, part, own, upto, of_wave);
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
        const int again = anew(pass);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            keys[mine[digit_of(k[u], again)] + rank_of(rank, u)] = k[u];
            if (u % 8 == 7) __builtin_amdgcn_sched_barrier(0);
        }
        unsigned before = 0;
        if (t < kRadix && tile > 0) {
            const unsigned* const p = look + t;
            int back = tile - 1, polls = 0;
            align_loop<K, T>();
            for (bool open = true; open;) {
                unsigned v[kWindow];
#pragma unroll
                for (int i = 0; i < kWindow; ++i)
                    v[i] = look_load(p + (size_t)(back >= i ? back - i : 0) * kRadix);
                bool ready = true;
                const int at = back;
#pragma unroll
                for (int i = 0; i < kWindow; ++i) {
                    ready = ready && (v[i] >> 30) != 0;
                    if (ready && open) {
                        before += v[i] & kLookCount;
                        open = (v[i] >> 30) != 2;  // tile 0's count is of all
                        --back;
                    }
                }
                // the tile before is running; the bound only ends a fault
                if (open && back == at && ++polls > kSpinLimit) {
                    __hip_atomic_fetch_or(a.ctr + CTR_ERROR * kWordStride, (int)ERR_SPIN_LIMIT, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
                    break;
                }
            }
            look_store(look + (size_t)tile * kRadix + t, kLookAll | (before + own));
        }
        if (t < kRadix) to[t] = start + before - upto;  // place of a key = to[digit] + its place in the tile
        __syncthreads();
        if (here == T && !split) {
            // eight at a time: all of them would take more registers than
            // the workgroups on a CU leave each other
            align_loop<K, T>();
#pragma unroll 1
            for (int u = 0; u < U; u += 8) {
#pragma unroll
                for (int v = 0; v < 8; ++v) {
                    const int i = (u + v) * kBulkThreads + t;
                    const K key = keys[i];
                    dst[to[digit_of(key, pass)] + (unsigned)i] = key;
                }
            }
        } else {
            for (int i = t; i < here; i += kBulkThreads) {
                const K key = keys[i];
                const int at = (int)to[digit_of(key, pass)] + i;
                if (split) *final_place(a, pl, at) = key;
                else dst[at] = key;
            }
        }
    }
}

// The heap's counters after a bulk call (one thread).
template <typename K>
__device__ __forceinline__ void set_counters(const BulkArgs<K>& a, const BulkPlan& pl) {
    a.ctr[CTR_BATCH_COUNT * kWordStride] = pl.nb_after;
    a.ctr[CTR_PARTIAL * kWordStride] = pl.pbs_after;
    if (a.calls > 0) a.ctr[CTR_DELETE_COUNT * kWordStride] = pl.off + pl.cut;
    a.ctr[CTR_ERROR * kWordStride] |= pl.error;
    const int busy = a.ctr[CTR_BUSY * kWordStride] + pl.busy;
    a.ctr[CTR_BUSY * kWordStride] = busy;
    if (pl.idle && busy <= 0) a.ctr[CTR_TERM * kWordStride] = 1;
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
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < kSortWords; i += 256) a.mem.hist[i] = 0;
    if (i0 == 0) set_counters(a, pl);
}

// A sort of one tile, whole: plan, passes in LDS, final places, counters.  The
// free slots are not used.
template <typename K>
__global__ __launch_bounds__(kBulkThreads, 2) void k_bulk_tile(BulkArgs<K> a) {
    constexpr int T = bulk_tile<K>(), U = T / kBulkThreads, W = kBulkThreads / 64, P = (int)sizeof(K);
    __shared__ K keys[T];
    __shared__ unsigned cnt[W][kRadix];
    __shared__ unsigned part[4];
    __shared__ BulkPlan pl;
    const int t = threadIdx.x, w = t >> 6, j = w * (64 * U) + (t & 63);
    if (t == 0) {
        plan_insert(a, pl);
        if (pl.total > T) pl.go = 0;
        *a.mem.plan = pl;
    }
    __syncthreads();
    if (!pl.go) return;
    const int total = pl.total;
    K k[U];
#pragma unroll 1
    for (int u = 0; u < U; ++u) keys[j + u * 64] = j + u * 64 < total ? *source_key(a, pl, j + u * 64) : ~K(0);
#pragma unroll
    for (int u = 0; u < U; ++u) k[u] = keys[j + u * 64];  // a thread reads back its own
#pragma unroll 1
    for (int pass = 0; pass < P; ++pass) {
        unsigned rank[U / 2];
#pragma unroll
        for (int i = 0; i < W * kRadix / kBulkThreads; ++i) (&cnt[0][0])[i * kBulkThreads + t] = 0;
        __syncthreads();
        rank_rows(k, pass, cnt[w], rank);
        __syncthreads();
        unsigned own = 0, upto = 0, of_wave[W];
        if (t < kRadix) count_digits(cnt, part, own, upto, of_wave);
        // (also the barrier before the sums and the counts are used)
        if (__syncthreads_or(own == (unsigned)T)) continue;  // the digit is the same for all
        if (t < kRadix) {
            for (int i = 0; i < w; ++i) upto += part[i];
#pragma unroll
            for (int i = 0; i < W; ++i) cnt[i][t] = upto + of_wave[i];
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < U; ++u) keys[cnt[w][digit_of(k[u], pass)] + rank_of(rank, u)] = k[u];
        __syncthreads();
#pragma unroll
        for (int u = 0; u < U; ++u) k[u] = keys[j + u * 64];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (j + u * 64 < total) *final_place(a, pl, j + u * 64) = k[u];
    const long long used = (pl.nb + 1ll) * a.batch_size;
    for (long long i = pl.fill_lo + t; i < used; i += kBulkThreads) a.items[i] = a.init_limits;
    for (int i = pl.pbs_after + t; i < a.batch_size; i += kBulkThreads) a.items[i] = a.init_limits;
    if (t == 0) set_counters(a, pl);
}

__global__ void k_bulk_report(const BulkPlan* pl, const int* ctr, int* report) {
    const int i = threadIdx.x;
    if (i <= CTR_WORDS) report[i] = i == 0 ? pl->go : ctr[(i - 1) * kWordStride];
}
static_assert(CTR_WORDS < kReportWords, "report words");

__global__ __launch_bounds__(256) void k_zero_words(int* status, long long nstatus, int* ctr, int nctr,
                                                    unsigned* sort, int nsort) {
    const long long i0 = blockIdx.x * 256ll + threadIdx.x, step = gridDim.x * 256ll;
    for (long long i = i0; i < nstatus; i += step) status[i] = 0;
    for (long long i = i0; i < nctr; i += step) ctr[i] = 0;
    for (long long i = i0; i < nsort; i += step) sort[i] = 0;
}

inline int blocks_for(long long items, int per_block, int most) {
    const long long b = (items + per_block - 1) / per_block;
    return (int)(b < 1 ? 1 : (b > most ? most : b));
}

// The last kernel of every call; its end is the event `done`.
template <typename K>
void finish(const BulkArgs<K>& a, long long keys, hipEvent_t done, int cus, hipStream_t s) {
    hipExtLaunchKernelGGL(k_bulk_finish<K>, dim3(blocks_for(keys, 4096, 8 * cus)), dim3(256), 0, s, nullptr, done, 0,
                          a);
}

// The sort of about `keys` keys; `mid`, if any, is recorded before the last
// pass, which hands the keys out.
template <typename K>
hipError_t sort_and_finish(const BulkArgs<K>& a, long long keys, hipEvent_t mid, hipEvent_t done, int cus,
                           hipStream_t s) {
    constexpr int P = (int)sizeof(K);
    hipLaunchKernelGGL(k_bulk_hist<K>, dim3(blocks_for(keys, 4096, 4 * cus)), dim3(256), 0, s, a);
    constexpr int kSmall = bulk_tile<K>(false), kLarge = bulk_tile<K>(true);
    const bool large = a.tile == kLarge;
    // two workgroups on a CU, also where three have room: the look-back gets
    // longer with every tile under way (2^24 u32 keys, 32 KB tiles: 324 us with
    // two, 353 with three, 363 with one and a half)
    const int grid = blocks_for(keys, a.tile, 2 * cus);
    for (int p = 0; p < P; ++p) {
        if (p == P - 1 && mid) {
            const hipError_t e = hipEventRecord(mid, s);
            if (e != hipSuccess) return e;
        }
        if (large) hipLaunchKernelGGL((k_bulk_pass<K, kLarge>), dim3(grid), dim3(kBulkThreads), 0, s, a, p);
        else hipLaunchKernelGGL((k_bulk_pass<K, kSmall>), dim3(grid), dim3(kBulkThreads), 0, s, a, p);
    }
    finish(a, keys, done, cus, s);
    return hipGetLastError();
}

template <typename K>
BulkArgs<K> args_for(const bgpq_heap* h, long long keys) {
    BulkArgs<K> a{};
    a.items = (K*)h->items;
    a.ctr = h->ctr;
    a.init_limits = (K)h->init_limits;
    a.batch_num = h->batch_num;
    a.batch_size = h->batch_size;
    a.tile = bulk_tile<K>(keys >= large_tiles_from<K>());
    a.mem = h->bulk;
    return a;
}

template <typename K>
hipError_t insert_as(const bgpq_heap* h, const void* keys, long long n, void* out, long long out_cap, long long calls,
                     int poppers, hipEvent_t mid, int cus, hipStream_t s) {
    BulkArgs<K> a = args_for<K>(h, h->held + n);
    a.keys = (const K*)keys;
    a.n = n;
    a.out = (K*)out;
    a.out_cap = out_cap;
    a.calls = calls;
    a.poppers = poppers;
    a.from_empty = mid != nullptr;
    clear_last_error();
    if (bulk_one_tile(h, h->held + n)) {
        if (mid) {
            const hipError_t e = hipEventRecord(mid, s);
            if (e != hipSuccess) return e;
        }
        hipExtLaunchKernelGGL(k_bulk_tile<K>, dim3(1), dim3(kBulkThreads), 0, s, nullptr, h->bulk_done, 0, a);
        return hipGetLastError();
    }
    return sort_and_finish(a, h->held + n, mid, h->bulk_done, cus, s);
}

template <typename K>
hipError_t delete_as(const bgpq_heap* h, void* out, long long out_cap, long long calls, int poppers, bool ascends,
                     int cus, hipStream_t s) {
    BulkArgs<K> a = args_for<K>(h, h->held);
    a.out = (K*)out;
    a.out_cap = out_cap;
    a.calls = calls;
    a.poppers = poppers;
    a.planned = 1;
    a.sorts = !ascends;
    clear_last_error();
    hipLaunchKernelGGL(k_plan_delete<K>, dim3(blocks_for(h->held / h->batch_size, 256, cus)), dim3(256), 0, s, a);
    hipLaunchKernelGGL(k_bulk_copy<K>, dim3(blocks_for(h->held, 8 * kBulkThreads, 4 * cus)), dim3(kBulkThreads), 0, s,
                       a);
    if (!ascends) return sort_and_finish(a, h->held, nullptr, h->bulk_done, cus, s);
    finish(a, h->held, h->bulk_done, cus, s);
    return hipGetLastError();
}

}  // namespace

hipError_t bulk_insert(const bgpq_heap* h, const void* keys, long long n, void* out, long long out_cap,
                       long long calls, int poppers, hipEvent_t mid, int cus, hipStream_t s) {
    return h->key_type == BGPQ_KEY_U64 ? insert_as<uint64_t>(h, keys, n, out, out_cap, calls, poppers, mid, cus, s)
                                       : insert_as<uint32_t>(h, keys, n, out, out_cap, calls, poppers, mid, cus, s);
}
bool bulk_one_tile(const bgpq_heap* h, long long keys) {
    return keys <= (h->key_type == BGPQ_KEY_U64 ? bulk_tile<uint64_t>() : bulk_tile<uint32_t>());
}
hipError_t zero_words(int* status, long long nstatus, int* ctr, int nctr, unsigned* sort, int nsort, hipStream_t s) {
    (void)hipGetLastError();  // report this launch only
    hipLaunchKernelGGL(k_zero_words, dim3(blocks_for(nstatus, 1024, 2048)), dim3(256), 0, s, status, nstatus, ctr, nctr,
                       sort, nsort);
    return hipGetLastError();
}
hipError_t bulk_report(const bgpq_heap* h, int* report, hipStream_t s) {
    hipLaunchKernelGGL(k_bulk_report, dim3(1), dim3(64), 0, s, h->bulk.plan, h->ctr, report);
    return hipGetLastError();
}
hipError_t bulk_delete(const bgpq_heap* h, void* out, long long out_cap, long long calls, int poppers, bool ascends,
                       int cus, hipStream_t s) {
    return h->key_type == BGPQ_KEY_U64 ? delete_as<uint64_t>(h, out, out_cap, calls, poppers, ascends, cus, s)
                                       : delete_as<uint32_t>(h, out, out_cap, calls, poppers, ascends, cus, s);
}

}  // namespace bgpq
