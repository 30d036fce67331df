"""Calls that carry many batches (insertions and deletions done together by
one radix sort, gpuheap_amd/csrc/bgpq_bulk.hpp) against the per-batch kernels
(a grid of one workgroup never bulks) and numpy: same keys out, same
counters, a heap the checker accepts and both kernels can go on with."""
import ctypes

import numpy as np
import pytest

import _oracle as O
import gpuheap_amd as G
from gpuheap_amd import DeviceBuffer, Heap, batch_num_for
from gpuheap_amd._lib import check, lib

pytestmark = pytest.mark.gpu

VARIANTS = list(G.VARIANTS)
PB = ("buitdd", "tditdd")


def _keys(key, n, seed, order):
    k = O.keys_u64(seed, n) if key == "u64" else O.keys_u32(seed, n)
    dt = k.dtype.type
    if order == "ascending":
        return np.sort(k)
    if order == "descending":
        return np.sort(k)[::-1].copy()
    if order == "ties":
        return (k % dt(12)) * dt(1000)
    if order == "one":
        return np.full(n, 77, k.dtype)
    if order == "byte2":  # one digit differs: every other pass is skipped
        return ((k % dt(256)) << dt(16)) + dt(3)
    return k


def _held(snapshot, B):
    """The keys of a heap in ascending order."""
    items, _, ctr = snapshot
    return np.sort(np.concatenate([items[:ctr[1]], items[B:B * (ctr[0] + 1)]]))


def _valid(h, keys):
    """The heap holds exactly these keys, in order for its checker."""
    assert h.checkInsertHeap(), h.last_check_message
    items, status, ctr = h.snapshot()
    B = h.batch_size
    assert not status.any() and ctr[3] == 0
    assert (ctr[0], ctr[1]) == (len(keys) // B, len(keys) % B)
    assert np.array_equal(_held((items, status, ctr), B), np.sort(keys))
    free = np.concatenate([items[ctr[1]:B], items[B * (ctr[0] + 1):]])
    assert (free == h.dtype.type(h.init_limits)).all(), "a free slot does not hold init_limits"


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("key,B", [("u32", 64), ("u32", 1024), ("u32", 8192), ("u64", 128), ("u64", 4096)])
@pytest.mark.parametrize("order", ["random", "ascending", "descending", "ties", "one", "byte2"])
def test_bulk_sort_orders(gpu, variant, key, B, order):
    # tiles of the passes hold 8192 u32 or 4096 u64 keys: counts around whole
    # tiles, the last tile one key, nearly full, full
    tile = 8192 if key == "u32" else 4096
    for n in (40 * tile, 40 * tile + 1, 43 * tile - 1):
        if variant not in PB:
            n = -(-n // B) * B
        n = max(n, 150 * B)
        print(f"[case] bulk {variant} {key} B={B} {order} n={n}", flush=True)
        keys = _keys(key, n, 5, order)
        h = Heap(batch_num_for(n, B), B, variant=variant, key=key)
        d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(keys.nbytes)
        h.insert(d, n)
        _valid(h, keys)
        h.delete(out, n // B + 1)
        G.sync()
        assert h.isEmpty() and h.error_flags() == 0
        assert np.array_equal(out.to_numpy(keys.dtype, n), np.sort(keys))
        _valid(h, keys[:0])
        h.close()


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("key", ["u32", "u64"])
def test_bulk_and_per_batch_calls_mixed(gpu, variant, key):
    """Bulk and per-batch calls on one heap in turn: bulk insertions into a
    heap the per-batch kernel filled and the reverse, partial drains of both
    kinds from ascending and from walked heaps; each pop equals the same
    calls on a heap driven by one workgroup."""
    B = 128
    pb = variant in PB
    rng = np.random.default_rng(3)
    a = Heap(4096, B, variant=variant, key=key)
    b = Heap(4096, B, variant=variant, key=key)
    cap = 1 << 20
    outs = [DeviceBuffer(cap * a.dtype.itemsize) for _ in range(2)]
    held = 0
    for step, (what, calls) in enumerate([("i", 3), ("i", 400), ("d", 2), ("d", 300), ("i", 5), ("i", 200), ("d", 150),
                                          ("d", 4), ("i", 900), ("d", 1), ("d", 700), ("i", 150), ("d", 5000)]):
        print(f"[case] bulk mixed {variant} {key} step {step} {what}{calls}", flush=True)
        if what == "i":
            chunk = int(rng.integers(B // 2, B + 1)) if pb else B
            n = calls * chunk - (int(rng.integers(1, chunk)) if pb else 0)
            keys = _keys(key, n, 100 + step, "ties" if step == 5 else "random")
            d = DeviceBuffer.from_numpy(keys)
            a.insert(d, n, chunk=chunk)
            b.insert(d, n, chunk=chunk, grid=1)
        else:
            a.delete(outs[0], calls)
            b.delete(outs[1], calls, grid=1)
        G.sync()
        assert a.checkInsertHeap(), a.last_check_message
        sa, sb = a.snapshot(), b.snapshot()
        assert np.array_equal(sa[2][:4], sb[2][:4])
        assert np.array_equal(_held(sa, B), _held(sb, B))
        done = sa[2][2]
        assert np.array_equal(outs[0].to_numpy(a.dtype, done), outs[1].to_numpy(a.dtype, done))
        # a few pops by one workgroup from the bulk heap's layout
        if what == "i":
            a.delete(outs[0], 2, grid=1)
            b.delete(outs[1], 2, grid=1)
            G.sync()
            assert a.checkInsertHeap(), a.last_check_message
    assert a.isEmpty() and b.isEmpty()


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("key", ["u32", "u64"])
@pytest.mark.parametrize("held,new,pops,room", [(0, 300, 200, 400), (200, 150, 350, 400), (200, 150, 500, 400),
                                                (250, 200, 300, 260), (300, 0, 290, 400), (120, 300, 0, 1)])
def test_bulk_concurrent(gpu, variant, key, held, new, pops, room):
    """A concurrent call: ascending pops, nothing lost, a valid heap left."""
    print(f"[case] bulk concurrent {variant} {key} held={held} new={new} pops={pops} room={room}", flush=True)
    B = 256
    part = 91 if variant in PB else 0  # a partial buffer, and another of 82 keys more
    n0, n1 = held * B + (part if held else 0), new * B + (part if new else 0)
    chunk = B // 2 if variant in PB else B
    keys = _keys(key, n0 + n1, held + pops, "random")
    h = Heap(1024, B, variant=variant, key=key)
    d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer((room * B + 5) * keys.itemsize)
    if n0:
        h.insert(d, n0)
    h.concurrent(d.ptr + n0 * keys.itemsize, n1, out, pops, chunk=chunk)
    G.sync()
    snap = h.snapshot()
    done = int(snap[2][2])
    batches, rest = divmod(n0 + n1, B)
    want = min(pops, batches, room) * B
    if pops > batches and room >= batches:
        want += rest
    assert done == want
    assert bool(snap[2][3] & 16) == (min(pops, batches) > room)
    got = out.to_numpy(keys.dtype, done)
    assert (got[1:] >= got[:-1]).all()
    left = _held(snap, B)
    assert np.array_equal(np.sort(np.concatenate([got, left])), np.sort(keys))
    if not snap[2][3]:
        assert h.checkInsertHeap(), h.last_check_message
    h.close()


@pytest.mark.parametrize("variant", VARIANTS)
def test_bulk_limits(gpu, variant):
    """What a bulk call must leave to the per-batch kernels or report like
    them: a heap without room for the sort's second buffer, one without room
    for the keys, an output that ends early, an init_limits below the type's
    largest, pointers not aligned to 16 bytes."""
    B, calls = 64, 600
    n = B * calls
    keys = O.keys_u32(21, n) >> np.uint32(1)
    d = DeviceBuffer.from_numpy(keys)
    print(f"[case] bulk limits {variant}: full heap", flush=True)
    h = Heap(calls, B, variant=variant, init_limits=1 << 31)
    h.insert(d, n)
    _valid(h, keys)
    h.insert(d, 300 * B)  # no slot left: overflow, nothing lost
    G.sync()
    assert h.error_flags() & 1 and h.nodeCount() == calls
    h.reset()
    h.insert(d, n)
    _valid(h, keys)
    out = DeviceBuffer(n * 4)
    h.delete(out, calls + 3)
    G.sync()
    assert h.isEmpty() and np.array_equal(out.to_numpy(np.uint32, n), np.sort(keys))
    print(f"[case] bulk limits {variant}: short output, odd alignment", flush=True)
    for spare in (0, 1):  # without and with room for a sort
        h = Heap(calls * (2 if spare else 1) + 2, B, variant=variant, init_limits=1 << 31)
        h.insert(d, n - B, grid=0)
        h.insert(d.ptr + 4 * (n - B), B, grid=1)
        h.set_cursor(3)
        room = 500 * B + 7
        out = DeviceBuffer(4 * n)
        mark = np.full(n, 0xABCDABCD, np.uint32)
        out.upload(mark)
        h.delete(out.ptr + 4, calls, out_keys=room)
        G.sync()
        assert h.error_flags() & 16
        got = out.to_numpy(np.uint32, n)
        m = (room - 3) // B * B
        assert np.array_equal(got[4:4 + m], np.sort(keys)[:m])
        assert (got[:4] == mark[0]).all() and (got[4 + m:] == mark[0]).all()
        assert h.itemCount() == n - m
        h.close()


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("key", ["u32", "u64"])
@pytest.mark.parametrize("order", ["random", "ties", "one", "byte2"])
def test_bulk_one_tile(gpu, variant, key, order):
    """Calls of one workgroup's sort (8192 u32, 4096 u64 keys and fewer): heap
    sorts of odd sizes around it, insertions into a heap that holds keys, and
    concurrent calls that leave some."""
    B, tile = 64, 8192 if key == "u32" else 4096
    for n in (20 * B, 20 * B + 1, tile - 1, tile, tile + 1):
        n = n if variant in PB else n // B * B
        print(f"[case] one tile {variant} {key} {order} n={n}", flush=True)
        keys = _keys(key, n, n, order)
        h = Heap(batch_num_for(n, B) + 64, B, variant=variant, key=key)
        d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(keys.nbytes)
        h.heapsort(d, n, d_out=out)
        assert np.array_equal(out.to_numpy(keys.dtype, n), np.sort(keys))
        _valid(h, keys[:0])
        h.insert(d, 19 * B)  # a bulk call, then more beside the keys held
        _valid(h, keys[:19 * B])
        h.set_cursor(0)
        m = n - 19 * B
        h.concurrent(d.ptr + 19 * B * keys.itemsize, m, out, 12, chunk=B)
        G.sync()
        done = int(h.snapshot()[2][2])
        assert done == min(12, n // B) * B
        if m // B >= 4:  # enough calls to be done together
            assert np.array_equal(out.to_numpy(keys.dtype, done), np.sort(keys)[:done])
            _valid(h, np.sort(keys)[done:])
        with pytest.raises(G.BgpqError, match="empty heap"):
            h.heapsort(d, B, d_out=out)
        h.close()


@pytest.mark.parametrize("key,B,n", [("u64", 1024, 1499999), ("u64", 1024, 1500000), ("u64", 4096, 184 * 8192 - 1),
                                     ("u64", 256, 184 * 8192), ("u64", 2048, 184 * 8192 + 1), ("u32", 1024, (1 << 22) - 1),
                                     ("u32", 1024, 1 << 22), ("u32", 512, (1 << 22) + 1), ("u32", 8192, 1 << 26),
                                     ("u32", 4096, (1 << 26) + 1), ("u32", 8192, (1 << 26) + 16383)])
@pytest.mark.parametrize("order", ["random", "byte2"])
def test_bulk_large_tiles(gpu, key, B, n, order):
    """Counts around the rule for the larger tiles and around whole ones."""
    print(f"[case] large tiles {key} B={B} n={n} {order}", flush=True)
    keys = _keys(key, n, n, order)
    want = np.sort(keys)
    h = Heap(batch_num_for(n, B), B, key=key)
    d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(keys.nbytes)
    h.heapsort(d, n, d_out=out)
    assert np.array_equal(out.to_numpy(keys.dtype, n), want)
    h.insert(d, n)
    h.set_cursor(0)
    h.delete(out, n // B // 3)
    h.delete(out, n // B + 1)
    G.sync()
    assert np.array_equal(out.to_numpy(keys.dtype, n), want)
    assert h.isEmpty() and h.error_flags() == 0
    h.close()


def test_bulk_needs_the_heap_to_itself(gpu):
    """After its view was handed out a heap takes the per-batch kernels only:
    the words of a walked heap differ from the ascending layout."""
    B, n = 64, 64 * 1000
    keys = O.keys_u32(4, n)
    d = DeviceBuffer.from_numpy(keys)

    def ascends(h):
        items = h.snapshot()[0][B:B * (n // B + 1)]
        return bool((items[1:] >= items[:-1]).all())

    h = Heap(4096, B)
    h.insert(d, n)
    assert ascends(h)
    g = Heap(4096, B)
    g.view()
    g.insert(d, n)
    assert not ascends(g) and g.checkInsertHeap()
    out = DeviceBuffer(n * 4)
    g.delete(out, n // B)
    G.sync()
    assert np.array_equal(out.to_numpy(np.uint32, n), np.sort(keys))


def test_bulk_calls_on_two_streams(gpu):
    """A call on another stream follows a bulk call on the first."""
    hip = ctypes.CDLL("libamdhip64.so")
    s = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
    B, n = 1024, 1 << 22
    keys = O.keys_u32(6, n)
    d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(n * 4)
    h = Heap(batch_num_for(n, B), B)
    h.insert(d, n)
    check(lib().bgpq_delete(h._h, out.ptr, n, n // B + 1, 0, s))
    assert hip.hipStreamSynchronize(s) == 0
    assert np.array_equal(out.to_numpy(np.uint32, n), np.sort(keys))
    assert h.isEmpty()
    h.close()
    assert hip.hipStreamDestroy(s) == 0


@pytest.mark.parametrize("same", [False, True])
def test_captured_calls_follow_a_bulk_call(gpu, same):
    """A call that is captured right behind a bulk call, on its stream or on
    another, is recorded as per-batch kernels; each replay acts on the heap it
    finds, with eager calls between."""
    print(f"[case] captured calls same={same}", flush=True)
    hip = ctypes.CDLL("libamdhip64.so")
    s, graph, run = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
    B, n = 256, 256 * 4000
    keys = O.keys_u32(9, n + B)
    d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(keys.nbytes)
    h = Heap(8192, B)
    a = Heap(64, B)  # loads what a first launch loads
    a.insert(d, B)
    a.delete(out, 1)
    a.view()
    a.insert(d, B)
    a.delete(out, 1)
    a.close()
    check(lib().bgpq_insert(h._h, d.ptr, n, 0, 0, s if same else None))
    assert hip.hipStreamBeginCapture(s, 0) == 0
    check(lib().bgpq_insert(h._h, d.ptr + 4 * n, B, 0, 0, s))
    check(lib().bgpq_delete(h._h, out.ptr, n, 2, 0, s))
    assert hip.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
    held, done = np.sort(keys[:n]), 0
    for i in range(4):
        assert hip.hipGraphLaunch(run, s) == 0
        assert hip.hipStreamSynchronize(s) == 0
        held = np.sort(np.concatenate([held, keys[n:]]))
        assert np.array_equal(out.to_numpy(np.uint32, done + 2 * B)[done:], held[:2 * B])
        held, done = held[2 * B:], done + 2 * B
        h.delete(out, 1, out_keys=n)  # eager
        G.sync()
        assert np.array_equal(out.to_numpy(np.uint32, done + B)[done:], held[:B])
        held, done = held[B:], done + B
        assert h.checkInsertHeap(), h.last_check_message
    assert h.itemCount() == len(held) and h.error_flags() == 0
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    h.close()
    assert hip.hipStreamDestroy(s) == 0


def test_view_follows_a_bulk_call(gpu):
    """A heap whose view is handed out right behind a bulk call is complete:
    a copy on a stream of its own finds the call's counters."""
    print("[case] view behind a bulk call", flush=True)
    hip = ctypes.CDLL("libamdhip64.so")
    s = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
    B, n = 1024, 1 << 26
    d = DeviceBuffer.from_numpy(O.keys_u32(12, n))
    h = Heap(batch_num_for(n, B), B)
    count = ctypes.c_int(-1)
    G.sync()
    h.insert(d, n)
    v = h.view()
    assert hip.hipMemcpyAsync(ctypes.byref(count), ctypes.c_void_p(v.ctr), ctypes.c_size_t(4), 2, s) == 0
    assert hip.hipStreamSynchronize(s) == 0
    assert count.value == n // B
    h.close()
    assert hip.hipStreamDestroy(s) == 0


@pytest.mark.parametrize("key,B,n", [("u32", 1024, 1 << 24), ("u64", 2048, 1 << 22), ("u32", 64, 1 << 12)])
def test_cursor_set_behind_a_bulk_insertion(gpu, key, B, n):
    """The output cursor set while a bulk insertion runs on a stream of its own
    stays: the insertion does not touch it, and the pops start there."""
    print(f"[case] cursor behind a bulk insertion {key} B={B} n={n}", flush=True)
    hip = ctypes.CDLL("libamdhip64.so")
    s = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
    keys = _keys(key, n, 14, "random")
    h = Heap(2 * batch_num_for(n, B) + 64, B, key=key)
    d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(8 * B * keys.itemsize)
    want = np.sort(keys)
    check(lib().bgpq_insert(h._h, d.ptr, n, 0, 0, s))
    check(lib().bgpq_delete(h._h, out.ptr, 8 * B, 5, 0, s))  # leaves the cursor at 5 B
    assert hip.hipStreamSynchronize(s) == 0
    assert h.snapshot()[2][2] == 5 * B
    check(lib().bgpq_insert(h._h, d.ptr, n, 0, 0, s))
    h.set_cursor(B)
    check(lib().bgpq_delete(h._h, out.ptr, 8 * B, 2, 0, s))
    assert hip.hipStreamSynchronize(s) == 0
    assert h.snapshot()[2][2] == 3 * B and h.error_flags() == 0
    held = np.sort(np.concatenate([want[5 * B:], want]))
    assert np.array_equal(out.to_numpy(keys.dtype, 3 * B)[B:], held[:2 * B])
    h.close()
    assert hip.hipStreamDestroy(s) == 0


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("B,batches,grid", [(64, 300, 32), (256, 100, 256), (1024, 40, 7)])
def test_bulk_pops_vote(gpu, variant, B, batches, grid):
    """Bulk pops take part in the termination vote as the per-batch kernels'
    workgroups do (counters 5 and 6: busy workgroups, the vote's end): on a
    heap whose view was handed out, and by the rule where only one answer is
    possible.  Not ended while workgroups are busy, ended once each of them has
    found nothing."""
    n = B * batches + (B // 2 if variant in PB else 0)
    got = -(-n // B)
    keys = O.keys_u32(batches, n)
    d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(keys.nbytes)
    for calls, busy, end in ((batches - 1, min(grid, batches - 1), 0), (got, min(grid, got), 0),
                             (got + 1, min(grid, got + 1) - 1, 0), (got + 8 * grid, 0, 1)):
        print(f"[case] vote {variant} B={B} batches={batches} grid={grid} calls={calls}", flush=True)
        for how in ("shared", "pops", "concurrent", "heapsort"):
            if how == "heapsort" and calls != got + 1:
                continue
            h = Heap(batch_num_for(n, B) + 64, B, variant=variant)
            if how == "shared":
                h.view()
            if how == "heapsort":
                h.heapsort(d, n, grid_delete=grid, d_out=out)
            elif how == "concurrent":
                h.concurrent(d, n, out, calls, grid=2 * grid, out_keys=n)
            else:
                h.insert(d, n)
                h.delete(out, calls, grid=grid, out_keys=n)
            G.sync()
            ctr = h.snapshot()[2]
            assert (ctr[5], ctr[6]) == (busy, end), how
            assert h.ifTerminate() == bool(end) and ctr[2] == min(calls * B, n)
            h.close()


@pytest.mark.parametrize("key,n,bits", [("u32", 1 << 26, 24), ("u32", 1 << 26, 9), ("u64", 1 << 24, 40)])
def test_delete_phase_hands_the_keys_out(gpu, key, n, bits):
    """A heap sort's delete phase holds the pass that hands the keys out also
    where the highest digits are the same for all keys and their passes are
    dropped.  That pass moves as many bytes as with all passes, so the phase
    takes about as long; without it, it would be the refill alone, a quarter."""
    print(f"[case] delete phase {key} n={n} bits={bits}", flush=True)
    B = 1024
    keys = _keys(key, n, 15, "random")
    few = keys >> keys.dtype.type(keys.itemsize * 8 - bits)
    h = Heap(batch_num_for(n, B), B, key=key)
    out = DeviceBuffer(keys.nbytes)
    ms = []
    for k in (keys, few):
        d = DeviceBuffer.from_numpy(k)
        ms.append(np.median([h.heapsort(d, n, d_out=out) for _ in range(7)], axis=0)[1])
        assert np.array_equal(out.to_numpy(k.dtype, n), np.sort(k))
        d.free()
    print(f"[case] delete phase {ms[0]:.3f} ms, {bits}-bit keys {ms[1]:.3f} ms", flush=True)
    assert ms[1] > 0.5 * ms[0]
    h.close()


@pytest.mark.parametrize("key", ["u32", "u64"])
def test_captured_reset(gpu, key):
    """A captured reset, insertion and pop: every replay starts from an empty
    heap, whatever eager calls did between."""
    print(f"[case] captured reset {key}", flush=True)
    hip = ctypes.CDLL("libamdhip64.so")
    s, graph, run = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
    B, n = 128, 128 * 20
    keys = _keys(key, n, 16, "random")
    d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(keys.nbytes)
    h = Heap(64, B, key=key)
    h.view()
    h.insert(d, n)  # loads what a first launch loads
    h.delete(out, 2)
    h.reset()
    G.sync()
    assert hip.hipStreamBeginCapture(s, 0) == 0
    check(lib().bgpq_reset(h._h, s))
    check(lib().bgpq_insert(h._h, d.ptr, n, 0, 0, s))
    check(lib().bgpq_delete(h._h, out.ptr, n, 3, 1, s))
    assert hip.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(run), graph, None, None, ctypes.c_size_t(0)) == 0
    want = np.sort(keys)
    for i in range(4):
        assert hip.hipGraphLaunch(run, s) == 0
        assert hip.hipStreamSynchronize(s) == 0
        _valid(h, want[3 * B:])
        assert h.snapshot()[2][2] == 3 * B
        assert np.array_equal(out.to_numpy(keys.dtype, 3 * B), want[:3 * B])
        h.insert(d, 5 * B - 7)  # eager
        h.delete(out, i)
        G.sync()
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    h.close()
    assert hip.hipStreamDestroy(s) == 0
