"""The drivers' loop where workgroups hold children and exchange them with the
root's batch: team sizes from one workgroup (which may never insert) to more
workgroups than batches, batch sizes with and without the split sift, both
partial-buffer variants; results equal the CPU oracles' and the heap is left
empty and valid."""
import numpy as np
import pytest

import _oracle as O
from gpuheap_amd import apps as A
from gpuheap_amd import Heap
from gpuheap_amd import serve as S

pytestmark = pytest.mark.gpu


def _heap(B, keys, variant):
    bn = 1
    while bn * B < 2 * keys + 128 * B:
        bn <<= 1
    return Heap(bn, B, variant=variant, key="u64")


@pytest.mark.parametrize("variant", ["buitdd", "tditdd"])
@pytest.mark.parametrize("B", [256, 512, 1024, 2048])
@pytest.mark.parametrize("grid", [1, 2, 7, 96])
def test_teams(gpu, variant, B, grid):
    print(f"[case] exchange {variant} B={B} grid={grid}: sssp", flush=True)
    rowptr, col, w = A.rmat_csr(13, 16, B + grid)
    with _heap(B, len(col), variant) as h:
        dist, st = A.sssp(h, A.Graph(rowptr, col, w), source=0, grid=grid)
        assert np.array_equal(dist, O.dijkstra(rowptr, col, w, 0))
        assert st["popped"] == st["expanded"] + st["stale"] == st["pushed"]
        assert h.isEmpty() and h.checkInsertHeap(), h.last_check_message
    print(f"[case] exchange {variant} B={B} grid={grid}: astar", flush=True)
    free = A.grid_map(311, 187, 0.25, B + grid)
    with _heap(B, 8 * 311 * 187, variant) as h:
        gm = A.GridMap(free, 311, 187)
        want, _ = O.astar(free, 311, 187)
        for _ in range(2):  # the second solve starts from the cleared heap
            cost, st = A.astar(h, gm, grid=grid)
            assert cost == want
            assert st["popped"] <= st["pushed"] and h.isEmpty()
    print(f"[case] exchange {variant} B={B} grid={grid}: knapsack", flush=True)
    w, v, cap = A.knapsack_instance(60, B + grid)
    with _heap(B, 1 << 18, variant) as h:
        best, st = A.knapsack(h, w, v, cap, grid=grid)
        assert best == O.knapsack_dp(w, v, cap)
        assert st["popped"] == st["expanded"] + st["stale"] + st["pruned"] == st["pushed"]
        assert h.isEmpty()


@pytest.mark.parametrize("team", [4, 6])
def test_children_and_partial_keys_over_two_batches(gpu, team):
    """Workgroups that hold nearly two batches of children when they take the
    partial buffer's keys in: none may be lost.  Which solves meet that depends
    on timing (5 in 1000 of these did), so many are run, each equal to the
    oracle bit for bit."""
    graphs = [A.rmat_csr(11, 16, 40 + i) for i in range(6)]
    dev = [A.Graph(*g) for g in graphs]
    qs, want, got = [], [], []
    for src in (0, 1, 2, 5):
        for g, d in zip(graphs, dev):
            want.append(O.dijkstra(*g, src))
            got.append(np.zeros(d.n, np.uint32))
            qs.append(S.sssp_query(d, src, batch_size=256, team=team, tag=len(qs), labels_out=got[-1]))
    budget = sum(S.query_bytes(q) + 4096 for q in qs)
    print(f"[case] exchange with partial keys team={team}", flush=True)
    for _ in range(100):
        res, _ = S.batch_run(qs, budget)
        for r, a, b in zip(res, got, want):
            assert r["status"] == 0 and np.array_equal(a, b)


@pytest.mark.parametrize("variant", ["buitdd", "tditdd"])
@pytest.mark.parametrize("B", [256, 2048])
def test_idle_workgroups_leave_together(gpu, variant, B):
    """Searches with one key at a time by 120 workgroups: most of them find
    nothing from their first pass to the last, and all waves of each must take
    the same way when the search ends."""
    print(f"[case] idle workgroups {variant} B={B}", flush=True)
    n = 40  # a path
    g = A.Graph(np.minimum(np.arange(n + 1), n - 1).astype(np.int32), np.arange(1, n, dtype=np.int32),
                np.full(n - 1, 3, np.uint32))
    free = np.ones(2 * 24, np.uint8)
    w, v, cap = A.knapsack_instance(12, 1)
    best, (cost, _) = O.knapsack_dp(w, v, cap), O.astar(free, 24, 2)
    with _heap(B, 1 << 14, variant) as h:
        for _ in range(10):
            dist, _ = A.sssp(h, g, source=0, grid=120)
            assert np.array_equal(dist, 3 * np.arange(n)) and h.isEmpty()
            assert A.astar(h, A.GridMap(free, 24, 2), grid=120)[0] == cost
            assert A.knapsack(h, w, v, cap, grid=120)[0] == best
