"""Which kernels do a call's work (Heap.route): the bulk sorts and copies, the
one-tile sort and the one-workgroup calls where a heap has itself to itself,
and one batch after the other wherever that does not hold or the heap refuses.
The answers of each are checked where the calls are tested; here, that the
tests meet the route they are about."""
import ctypes

import numpy as np
import pytest

import _oracle as O
import gpuheap_amd as G
from gpuheap_amd import DeviceBuffer, Heap, batch_num_for
from gpuheap_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def _keys(key, n):
    return O.keys_u64(n, n) if key == "u64" else O.keys_u32(n, n)


def _digits(keys):
    """Bytes in which the keys differ: the passes that must move them."""
    return int((np.ptp(keys.view(np.uint8).reshape(len(keys), -1), axis=0) > 0).sum())


@pytest.mark.parametrize("variant", list(G.VARIANTS))
@pytest.mark.parametrize("key,B,single", [("u32", 64, True), ("u32", 1024, True), ("u32", 4096, True),
                                          ("u32", 8192, False), ("u64", 64, True), ("u64", 512, True),
                                          ("u64", 1024, False), ("u64", 4096, False)])
def test_single_calls_take_one_workgroup(gpu, variant, key, B, single):
    print(f"[case] route of single calls {variant} {key} B={B}", flush=True)
    want = ("single" if single else "batches", 0)
    keys = _keys(key, 4 * B)
    h = Heap(3, B, variant=variant, key=key)
    d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(keys.nbytes)
    for i in range(3):
        h.insert(d.ptr + i * B * keys.itemsize, B)
        assert h.route() == want
    h.delete(out, 1, out_keys=B - 1)  # an output that ends early
    assert h.route() == ("batches", 0) and h.error_flags() & 16
    h.delete(out, 1)
    assert h.route() == want
    h.delete(out, 1, grid=1)
    assert h.route() == ("batches", 0)
    h.delete(out, 1)
    assert h.route() == want and h.isEmpty()
    h.delete(out, 1)  # nothing to pop
    assert h.route() == ("batches", 0)
    assert np.array_equal(out.to_numpy(keys.dtype, 3 * B), np.sort(keys[:3 * B]))
    if not variant.endswith("_np"):
        h.insert(d, B - 1)  # a first partial batch
        assert h.route() == ("batches", 0)
    h.close()


@pytest.mark.parametrize("variant", list(G.VARIANTS))
@pytest.mark.parametrize("key", ["u32", "u64"])
def test_many_batches_are_sorted(gpu, variant, key):
    print(f"[case] route of many batches {variant} {key}", flush=True)
    B, tile = 64, 8192 if key == "u32" else 4096
    n = 300 * B
    keys = _keys(key, n)
    passes = _digits(keys)  # u64 keys end in their index: below 2^16 here
    assert passes == (4 if key == "u32" else 6)
    h = Heap(700, B, variant=variant, key=key)
    d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(keys.nbytes)
    h.insert(d, tile // 2)
    assert h.route() == ("tile", 0)
    h.concurrent(d, tile // 2, out, 10)
    assert h.route() == ("tile", 0)
    h.delete(out, 30)
    assert h.route() == ("copy", 0)
    h.clear()
    h.insert(d, n)
    assert h.route() == ("sort", passes)
    h.set_cursor(0)
    h.delete(out, 1)  # a walk: the slots ascend no more
    assert h.route() == ("single", 0)
    h.delete(out, 100)
    assert h.route() == ("sort", passes)
    h.delete(out, 100)
    assert h.route() == ("copy", 0)
    h.concurrent(d, 150 * B, out, 100, out_keys=n)
    assert h.route() == ("sort", passes)
    h.clear()
    h.heapsort(d, tile, d_out=out)
    assert h.route() == ("tile", 0)
    h.heapsort(d, n, d_out=out)
    assert h.route() == ("sort", passes)
    few = DeviceBuffer.from_numpy(keys % keys.dtype.type(200) << keys.dtype.type(16))
    h.heapsort(few, n, d_out=out)  # one digit differs: two passes, the fewest
    assert h.route() == ("sort", 2)
    h.close()


@pytest.mark.parametrize("key,B,n", [("u64", 1024, 1500000), ("u32", 1024, 1 << 22)])
def test_large_sorts(gpu, key, B, n):
    print(f"[case] route of a large sort {key} n={n}", flush=True)
    keys = _keys(key, n)
    h = Heap(batch_num_for(n, B), B, key=key)
    d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(keys.nbytes)
    h.heapsort(d, n, d_out=out)
    assert h.route()[0] == "sort"
    h.insert(d, n)
    assert h.route()[0] == "sort"
    h.set_cursor(0)
    h.delete(out, n // B + 1)
    assert h.route() == ("copy", 0)
    h.close()


def test_batches_where_the_heap_is_shared_or_full(gpu):
    print("[case] route of shared and full heaps", flush=True)
    hip = ctypes.CDLL("libamdhip64.so")
    B, n = 64, 64 * 400
    keys = O.keys_u32(3, n + 1)
    d, out = DeviceBuffer.from_numpy(keys), DeviceBuffer(keys.nbytes)
    per_batch = ("batches", 0)
    h = Heap(401, B)
    h.insert(d, n)  # no room for the sort's second buffer
    assert h.route() == per_batch
    h.insert(d, 100 * B)  # nor for the keys
    assert h.route() == per_batch and h.error_flags() & 1
    h.close()
    h = Heap(1024, B)
    h.insert(d, n, grid=1)
    assert h.route() == per_batch
    h.delete(out.ptr + 2, 100, out_keys=n)  # not aligned to the keys' size
    assert h.route() == per_batch
    h.reset()
    h.view()
    h.insert(d, n)
    assert h.route() == per_batch
    h.delete(out, 1)
    assert h.route() == per_batch
    h.close()
    s = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
    h = Heap(1024, B)
    h.insert(d, n)
    assert h.route()[0] == "sort"
    check(lib().bgpq_delete(h._h, out.ptr, n, 100, 0, s))
    assert h.route() == per_batch
    h.close()
    assert hip.hipStreamDestroy(s) == 0
