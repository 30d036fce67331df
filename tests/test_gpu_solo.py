"""Single insertions and pops on a heap that has itself to itself (one workgroup
without locks, gpuheap_amd/csrc/bgpq_solo.hip): every state it can meet (empty,
one batch, partial buffers filled and folded, a full heap, a short output),
heaps the checker accepts after each call, and the smallest keys out."""
import ctypes

import numpy as np
import pytest

import _oracle as O
import gpuheap_amd as G
from gpuheap_amd import DeviceBuffer, Heap
from gpuheap_amd._lib import check, lib

pytestmark = pytest.mark.gpu

VARIANTS = list(G.VARIANTS)
PB = ("buitdd", "tditdd")
SIZES = [("u32", 64), ("u32", 256), ("u32", 1024), ("u32", 4096), ("u64", 64), ("u64", 256), ("u64", 512)]


def _state(h, held):
    assert h.checkInsertHeap(), h.last_check_message
    items, status, ctr = h.snapshot()
    B = h.batch_size
    assert not status.any() and ctr[0] * B + ctr[1] == len(held)
    assert np.array_equal(np.sort(np.concatenate([items[:ctr[1]], items[B:B * (ctr[0] + 1)]])), held)
    assert (np.concatenate([items[ctr[1]:B], items[B * (ctr[0] + 1):]]) == h.dtype.type(h.init_limits)).all()
    return ctr


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("key,B", SIZES)
@pytest.mark.parametrize("order", ["random", "ascending", "descending", "ties"])
def test_single_calls(gpu, variant, key, B, order):
    print(f"[case] single calls {variant} {key} B={B} {order}", flush=True)
    rng = np.random.default_rng(B)
    cap = 21
    n = 64 * B
    keys = O.keys_u64(B, n) if key == "u64" else O.keys_u32(B, n)
    if order == "ties":
        keys = keys % keys.dtype.type(7)
    elif order != "random":
        keys = np.sort(keys)
        keys = keys if order == "ascending" else keys[::-1].copy()
    h = Heap(cap, B, variant=variant, key=key)
    d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(keys.nbytes)
    ks, held, at, done = keys.itemsize, keys[:0], 0, 0
    # up to a nearly full heap, down to an empty one, and up again
    for step in range(64):
        push = step < 24 if step < 44 else step % 3 != 0
        if push and len(held) + B <= cap * B:
            m = B if variant not in PB or rng.random() < 0.5 else int(rng.integers(1, B + 1))
            if at + m > n:
                break
            h.insert(d.ptr + at * ks, m)
            held = np.sort(np.concatenate([held, keys[at:at + m]]))
            at += m
        else:
            h.delete(out, 1)
            m = min(B, len(held)) if variant in PB else (B if len(held) else 0)
            G.sync()
            assert np.array_equal(out.to_numpy(keys.dtype, done + m)[done:], held[:m])
            held, done = held[m:], done + m
        G.sync()
        assert _state(h, held)[2] == done
    assert h.error_flags() == 0
    h.close()


@pytest.mark.parametrize("variant", VARIANTS)
def test_single_call_limits(gpu, variant):
    """Calls that the general kernels report: a full heap, an output that ends
    early, nothing to pop; and an output and keys that are not aligned to 16
    bytes."""
    print(f"[case] single call limits {variant}", flush=True)
    B, cap = 128, 5
    keys = O.keys_u32(3, (cap + 2) * B + 1)
    d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(keys.nbytes)
    h = Heap(cap, B, variant=variant)
    h.delete(out, 1)
    G.sync()
    assert h.isEmpty() and h.error_flags() == 0
    for i in range(cap):
        h.insert(d.ptr + 4 * (1 + i * B), B)
    h.insert(d.ptr + 4 * (1 + cap * B), B)
    held = np.sort(keys[1:1 + cap * B])
    G.sync()
    assert h.error_flags() & 1 and h.nodeCount() == cap
    h.delete(out.ptr + 4, 1, out_keys=2 * B - 1)
    h.delete(out.ptr + 4, 1, out_keys=2 * B - 1)
    G.sync()
    assert h.error_flags() & 16 and h.nodeCount() == cap - 1
    assert np.array_equal(out.to_numpy(np.uint32, B + 1)[1:], held[:B])
    h.close()


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("key,B,cap", [("u32", 64, 9), ("u32", 256, 12), ("u64", 128, 13), ("u32", 4096, 5)])
@pytest.mark.parametrize("above", [False, True])
def test_single_pops_stay_in_the_slots(gpu, variant, key, B, cap, above):
    """Keys at init_limits and above it, which no caller may insert: a pop whose
    node has a left child only goes down to that one, never to a slot past the
    last.  Every key comes out, and no free slot is written."""
    print(f"[case] keys at the limit {variant} {key} B={B} cap={cap} above={above}", flush=True)
    limit = (1 << 32) - 1 if not above else 1 << 31
    n = cap * B
    keys = O.keys_u64(cap, n) >> np.uint64(32) if key == "u64" else O.keys_u32(cap, n)
    if not above:
        keys[keys > keys.dtype.type(1 << 31)] = limit
    h = Heap(cap, B, init_limits=limit, variant=variant, key=key)
    d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(keys.nbytes)
    for i in range(cap):
        h.insert(d.ptr + i * B * keys.itemsize, B)
    G.sync()
    want = np.sort(keys)
    for i in range(cap):
        h.delete(out, 1)
        G.sync()
        items, status, ctr = h.snapshot()
        assert (ctr[0], ctr[1], ctr[2], ctr[3]) == (cap - i - 1, 0, (i + 1) * B, 0) and not status.any()
        assert np.array_equal(np.sort(items[B:B * (cap - i)]), want[(i + 1) * B:])
        assert (items[B * (cap - i):] == keys.dtype.type(limit)).all()
    assert np.array_equal(out.to_numpy(keys.dtype, n), want)
    h.close()


def test_single_calls_on_two_streams(gpu):
    """A single call on another stream follows one on the first."""
    hip = ctypes.CDLL("libamdhip64.so")
    s = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
    B = 4096
    keys = O.keys_u32(8, 4 * B)
    d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(keys.nbytes)
    h = Heap(64, B)
    for i in range(4):
        h.insert(d.ptr + 4 * i * B, B)
    check(lib().bgpq_delete(h._h, out.ptr, 4 * B, 4, 0, s))
    assert hip.hipStreamSynchronize(s) == 0
    assert np.array_equal(out.to_numpy(np.uint32, 4 * B), np.sort(keys)) and h.isEmpty()
    h.close()
    assert hip.hipStreamDestroy(s) == 0
