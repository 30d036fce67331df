"""Timed cases of the heap: what a user's program has it do, through the
public Python entry points (Heap, apps, serve.batch_run).

A case is a dict of plain values; ``kind`` says which path it takes:

sort      Heap.heapsort of n device keys into a second buffer: every key
          inserted, then popped until the heap is empty
harness   the reference's harness: insert the lower half of the keys in
          partial chunks, insert the upper half while the lower is popped,
          pop the rest
stream    a running queue: rounds of bulk insertions and bulk pops on one
          heap that stays partly filled, then a drain
hold      pop one batch from a filled heap and push it back (the smallest
          calls the heap has)
sssp      Dijkstra's frontier on an R-MAT graph, distances fetched
astar     an 8-connected obstacle grid, corner to corner
knapsack  0/1 branch and bound
batch     many independent solves at once, each on a heap of its own

Keys are uniform (or ordered) as in the heap-sort sweep, graphs are R-MAT
with a, b, c = 0.57, 0.19, 0.19 and weights 1..1000, grids have obstacle
density 0.25, knapsack values are weight + 100 with half the total weight as
capacity: the distributions the benchmark and the tests use.
"""
import math

import numpy as np
import torch

import gpuheap_amd as G
from gpuheap_amd import apps as A
from gpuheap_amd import serve as S

VARIANTS = ("buitdd", "buitdd_np", "tditdd", "tditdd_np")
KEY_BYTES = {"u32": 4, "u64": 8}
INF = 0xFFFFFFFF


def listed():
    return [
        # a few batches, ragged: launches and latency
        dict(name="sort_small", kind="sort", n=3001, B=256, variant="buitdd", key="u32", order="random", gi=0, gd=0),
        # the plain heap sort: 2^20 keys at B = 1024
        dict(name="sort_1m", kind="sort", n=1 << 20, B=1024, variant="buitdd", key="u32", order="random", gi=0, gd=0),
        # the adversarial order, full batches only
        dict(name="sort_desc", kind="sort", n=6001 * 2048, B=2048, variant="tditdd_np", key="u32", order="descending",
             gi=256, gd=64),
        # 32-bit keys with a 32-bit payload, ragged
        dict(name="sort_u64", kind="sort", n=3000017, B=1024, variant="tditdd", key="u64", order="random", gi=0, gd=0),
        # the headline workload
        dict(name="sort_2p28", kind="sort", n=1 << 28, B=8192, variant="buitdd_np", key="u32", order="random", gi=256,
             gd=64),
        # insert, insert beside pops, pop: partial chunks at the harness's grid
        dict(name="harness_1m", kind="harness", n=1 << 20, B=512, variant="buitdd", key="u32", grid=32),
        # a running queue of (priority, payload) keys
        dict(name="stream_u64", kind="stream", n=1500000, rounds=6, B=1024, variant="buitdd", key="u64"),
        # one pop and one push on a filled heap
        dict(name="hold_u64", kind="hold", n=1 << 20, B=256, variant="buitdd", key="u64"),
        # single solves with the workgroup counts the drivers run best at
        dict(name="sssp_18", kind="sssp", scale=18, B=1024, grid=32),
        dict(name="astar_1024", kind="astar", width=1024, height=1024, B=256, grid=4),
        dict(name="knapsack_200", kind="knapsack", items=200, B=256, grid=8),
        # the mixed workload's shares and sizes, solved at once
        dict(name="batch_mixed", kind="batch", queries=60, max_scale=14, max_side=512),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sort"] * 5 + ["harness", "stream", "stream", "hold", "sssp", "astar", "knapsack", "batch"])
    key = rng.choice(["u32", "u32", "u64"])
    variant = rng.choice(VARIANTS)
    B = rng.choice([128, 256, 512, 1024, 2048, 4096, 8192])
    if key == "u64":
        B = min(B, 4096)
    if kind == "sort":
        n = _log_int(rng, 1000, min(1 << 27, B << 13))
        if variant.endswith("_np"):
            n = max(n // B, 1) * B
        gi, gd = rng.choice([(0, 0), (256, 64), (32, 32)])
        order = rng.choice(["random", "random", "random", "descending", "ascending", "ties"])
        return dict(kind=kind, n=n, B=B, variant=variant, key=key, order=order, gi=gi, gd=gd)
    if kind == "harness":
        B = min(B, 2048)
        n = _log_int(rng, 16 * B, 2048 * B)
        if variant.endswith("_np"):
            n = max(n // (2 * B), 1) * 2 * B
        return dict(kind=kind, n=n, B=B, variant=variant, key=key, grid=rng.choice([32, 64, 128]))
    if kind == "stream":
        n = _log_int(rng, 16 * B, min(1 << 24, 4096 * B))
        return dict(kind=kind, n=n, rounds=rng.randint(2, 10), B=B, variant=variant, key=key)
    if kind == "hold":
        n = _log_int(rng, 8 * B, 4096 * B)
        return dict(kind=kind, n=n, B=B, variant=variant, key=key)
    if kind == "sssp":
        return dict(kind=kind, scale=rng.randint(10, 19), B=rng.choice([256, 512, 1024, 2048]),
                    grid=rng.choice([8, 16, 32, 64]))
    if kind == "astar":
        w = _log_int(rng, 100, 1200)
        return dict(kind=kind, width=w, height=max(64, int(w * rng.uniform(0.6, 1.2))), B=rng.choice([256, 512]),
                    grid=rng.choice([1, 2, 4, 8]))
    if kind == "knapsack":
        return dict(kind=kind, items=rng.randint(40, 200), B=rng.choice([256, 512]), grid=rng.choice([4, 8, 16]))
    return dict(kind="batch", queries=rng.randint(5, 60), max_scale=rng.randint(11, 14),
                max_side=rng.choice([256, 384, 512]))


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _values(case, seed):
    """The case's keys as int64 values in input order."""
    n, g = case["n"], _gen(seed)
    order = case.get("order", "random")
    k = torch.randint(0, 12 if order == "ties" else INF, (n,), generator=g, device="cuda", dtype=torch.int64)
    if order == "ties":
        k *= 1000
    if case["kind"] == "harness":  # the keys inserted beside the pops lie above all others
        half = _half(case)
        k >>= 1
        k[half:] += 1 << 31
        k.clamp_(max=INF - 1)
    if order in ("ascending", "descending"):
        k = torch.sort(k, descending=order == "descending").values
    if case["key"] == "u64":  # payload: the input position (priorities of 31 bits keep int64's sign)
        k = ((k >> 1) << 32) | torch.arange(n, device="cuda", dtype=torch.int64)
    return k


def _keys(case, values):
    """Values as the heap's unsigned keys: their bits in an integer tensor of
    the keys' width (u32 keys from 2^31 on show as negative int32)."""
    return values.clone() if case["key"] == "u64" else values.to(torch.int32)


def _dtype(case):
    return torch.int64 if case["key"] == "u64" else torch.int32


def _half(case):
    unit = case["B"] if case["variant"].endswith("_np") else 1
    return case["n"] // 2 // unit * unit


def _rounds(case):
    """Per round of a stream: (first key, keys inserted, batches popped).
    The queue grows in the first rounds and keeps a backlog until the end."""
    n, r, B = case["n"], case["rounds"], case["B"]
    np_ = case["variant"].endswith("_np")
    out, at = [], 0
    for i in range(r):
        m = n // r
        if np_:
            m = m // B * B
        out.append((at, m, (m * (i + 1) // (r + 1)) // B))
        at += m
    return out


def _heap(case, n):
    return G.Heap(G.batch_num_for(n, case["B"]), case["B"], variant=case["variant"], key=case["key"])


def _rmat(scale, seed, degree=16):
    g = _gen(seed)
    ne = degree << scale
    src = torch.zeros(ne, dtype=torch.int64, device="cuda")
    dst = torch.zeros(ne, dtype=torch.int64, device="cuda")
    for _ in range(scale):
        r = torch.rand(ne, generator=g, device="cuda")
        src = src * 2 + (r >= 0.76)
        dst = dst * 2 + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    w = torch.randint(1, 1001, (ne,), generator=g, device="cuda", dtype=torch.int64)
    order = torch.argsort(src, stable=True)
    src, dst, w = src[order], dst[order], w[order]
    row = torch.zeros((1 << scale) + 1, dtype=torch.int64, device="cuda")
    row[1:] = torch.cumsum(torch.bincount(src, minlength=1 << scale), 0)
    return row, src, dst, w


def _graph(scale, seed):
    row, _, dst, w = _rmat(scale, seed)
    return A.Graph(row.cpu().numpy().astype(np.int32), dst.cpu().numpy().astype(np.int32),
                   w.cpu().numpy().astype(np.uint32))


def _grid(width, height, seed):
    free = (torch.rand(width * height, generator=_gen(seed), device="cuda") >= 0.25).to(torch.uint8)
    free[0] = free[-1] = 1
    return free


def _items(n, seed):
    w = np.random.default_rng(seed).integers(1, 1001, size=n).astype(np.uint32)
    return w, (w + 100).astype(np.uint32), int(w.sum()) // 2


def _bn(keys, B):
    bn = 1
    while bn * B < keys + 16 * B:
        bn <<= 1
    return bn


def _queries(case, seed):
    """(kind, size, seed of its input) of a batch: 40% SSSP on 2^10..2^max
    vertices, 40% A* on 256^2..max^2 cells, 20% knapsack.  The sizes belong to
    the case, the inputs to the seed."""
    rng = np.random.default_rng(case["queries"])
    q = []
    for i in range(case["queries"]):
        s = (seed * 1000 + i) % (1 << 40)
        if i % 5 < 2:
            q.append(("sssp", 10 + int(rng.integers(case["max_scale"] - 9)), s))
        elif i % 5 < 4:
            q.append(("astar", int(round(256 * (case["max_side"] / 256) ** rng.random())), s))
        else:
            q.append(("knapsack", 200, s))
    return q


# ----------------------------------------------------------------- prepare
def prepare(case, seed):
    kind, B = case["kind"], case.get("B")
    if kind in ("sort", "harness", "stream", "hold"):
        n = case["n"]
        st = dict(case=case, keys=_keys(case, _values(case, seed)), heap=_heap(case, n))
        st["out"] = torch.empty(B if kind == "hold" else n, dtype=_dtype(case), device="cuda")
        torch.cuda.synchronize()
        if kind == "hold":
            m = n // B * B  # whole batches, so that a pop takes one
            st["heap"].insert(st["keys"].data_ptr(), m)
            G.sync()
        return st
    if kind == "sssp":
        g = _graph(case["scale"], seed)
        return dict(case=case, graph=g, heap=A.app_heap(B, _bn(g.m, B)))
    if kind == "astar":
        w, h = case["width"], case["height"]
        m = A.GridMap(_grid(w, h, seed).cpu().numpy(), w, h)
        return dict(case=case, map=m, heap=A.app_heap(B, _bn(4 * w * h, B)))
    if kind == "knapsack":
        return dict(case=case, items=_items(case["items"], seed), heap=A.app_heap(B, _bn(1 << 20, B)))
    qs, inputs, answers = [], [], []
    for i, (what, size, s) in enumerate(_queries(case, seed)):
        if what == "sssp":
            g = _graph(size, s)
            inputs.append(g)
            labels = np.empty(g.n, np.uint32)
            qs.append(S.sssp_query(g, 0, batch_size=1024, team=4, tag=i, labels_out=labels))
            answers.append(labels)
        elif what == "astar":
            g = A.GridMap(_grid(size, size, s).cpu().numpy(), size, size)
            inputs.append(g)
            qs.append(S.astar_query(g, batch_size=256, team=2, tag=i))
            answers.append(None)
        else:
            qs.append(S.knapsack_query(*_items(size, s), batch_size=256, team=2, tag=i))
            answers.append(None)
    budget = sum(S.query_bytes(q) + 4096 for q in qs)
    return dict(case=case, queries=qs, inputs=inputs, answers=answers, budget=budget)


# --------------------------------------------------------------------- run
def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "sort":
        state["heap"].heapsort(state["keys"].data_ptr(), c["n"], grid_insert=c["gi"], grid_delete=c["gd"],
                               d_out=state["out"].data_ptr())
        return state["out"]
    if kind == "harness":
        h, n, B, half = state["heap"], c["n"], c["B"], _half(c)
        np_ = c["variant"].endswith("_np")
        src, dst = state["keys"].data_ptr(), state["out"].data_ptr()
        calls = (half + B - 1) // B
        h.set_cursor(0)
        h.insert(src, half, chunk=B if np_ else B // 3, grid=c["grid"])
        h.concurrent(src + half * KEY_BYTES[c["key"]], n - half, dst, calls, chunk=B if np_ else 2 * B // 3,
                     grid=c["grid"], out_keys=n)
        h.delete(dst, (n - half + B - 1) // B + 1, grid=c["grid"], out_keys=n)
        return state["out"]
    if kind == "stream":
        h, B, ks = state["heap"], c["B"], KEY_BYTES[c["key"]]
        src, dst, n = state["keys"].data_ptr(), state["out"].data_ptr(), c["n"]
        h.set_cursor(0)
        for at, m, pops in _rounds(c):
            h.insert(src + at * ks, m)
            h.delete(dst, pops, out_keys=n)
        h.delete(dst, n // B + 1, out_keys=n)
        return state["out"][:sum(m for _, m, _ in _rounds(c))]
    if kind == "hold":
        h = state["heap"]
        p = state["out"].data_ptr()
        h.set_cursor(0)
        h.delete(p, 1, out_keys=c["B"])
        h.insert(p, c["B"])
        return state["out"]
    if kind == "sssp":
        return A.sssp(state["heap"], state["graph"], 0, grid=c["grid"])[0]
    if kind == "astar":
        return A.astar(state["heap"], state["map"], grid=c["grid"])[0]
    if kind == "knapsack":
        return A.knapsack(state["heap"], *state["items"], grid=c["grid"])[0]
    res, _ = S.batch_run(state["queries"], state["budget"])
    # an SSSP's distances, an A* cost, a knapsack value
    return [r["value"] if a is None else a for r, a in zip(res, state["answers"])]


# -------------------------------------------------------------------- work
def work(case):
    """Bytes each input and output takes once; no floating-point work."""
    kind = case["kind"]
    if kind in ("sort", "harness"):
        b = 2 * case["n"] * KEY_BYTES[case["key"]]
    elif kind == "stream":
        b = 2 * sum(m for _, m, _ in _rounds(case)) * KEY_BYTES[case["key"]]
    elif kind == "hold":
        b = 4 * case["B"] * KEY_BYTES[case["key"]]  # popped and pushed: read and written once each
    elif kind == "sssp":
        b = _sssp_bytes(case["scale"])
    elif kind == "astar":
        b = 5 * case["width"] * case["height"]  # the map and one label a cell
    elif kind == "knapsack":
        b = 8 * case["items"]
    else:
        b = 0
        for what, size, _ in _queries(case, 0):
            b += _sssp_bytes(size) if what == "sssp" else 5 * size * size if what == "astar" else 8 * size
    return {"bytes": b, "flops": 0}


def _sssp_bytes(scale):
    return (8 << scale) + (16 << scale) * 8  # row offsets and distances; targets and weights


# ------------------------------------------------------------------- exact
def exact(case, seed):
    kind = case["kind"]
    if kind in ("sort", "harness"):
        return _keys(case, torch.sort(_values(case, seed)).values)
    if kind == "hold":
        m = case["n"] // case["B"] * case["B"]
        return _keys(case, torch.sort(_values(case, seed)[:m]).values[:case["B"]])
    if kind == "stream":
        v, B = _values(case, seed), case["B"]
        held, out = v[:0], []
        for at, m, pops in _rounds(case):
            held = torch.sort(torch.cat([held, v[at:at + m]])).values
            take = min(pops, len(held) // B) * B
            out.append(held[:take])
            held = held[take:]
        return _keys(case, torch.cat(out + [held]))
    if kind == "sssp":
        return _distances(*_rmat(case["scale"], seed))
    if kind == "astar":
        return _path_cost(_grid(case["width"], case["height"], seed), case["width"], case["height"])
    if kind == "knapsack":
        return _best_value(*_items(case["items"], seed))
    out = []
    for what, size, s in _queries(case, seed):
        if what == "sssp":
            out.append(_distances(*_rmat(size, s)))
        elif what == "astar":
            out.append(_path_cost(_grid(size, size, s), size, size))
        else:
            out.append(_best_value(*_items(size, s)))
    return out


def _distances(row, src, dst, w):
    """Distances from vertex 0 by rounds of relaxation over all edges."""
    d = torch.full((len(row) - 1,), 1 << 40, dtype=torch.int64, device=row.device)
    d[0] = 0
    while True:
        e = d.scatter_reduce(0, dst, d[src] + w, "amin")
        if torch.equal(e, d):
            break
        d = e
    return torch.where(d >= 1 << 39, INF, d).cpu().numpy().astype(np.uint32)


def _path_cost(free, width, height):
    """Cost from the first cell to the last by rounds of relaxation."""
    big = 1 << 40
    blocked = torch.full((height + 2, width + 2), big, dtype=torch.int64, device=free.device)
    blocked[1:-1, 1:-1][free.view(height, width) != 0] = 0
    d = torch.full_like(blocked, big)
    d[1, 1] = 0
    while True:
        last = d.clone()
        for _ in range(32):
            e = d.clone()
            for dy in (-1, 0, 1):
                for dx in (-1, 0, 1):
                    if dx or dy:
                        step = 14 if dx and dy else 10
                        near = d[1 + dy:height + 1 + dy, 1 + dx:width + 1 + dx] + step
                        e[1:-1, 1:-1] = torch.minimum(e[1:-1, 1:-1], near + blocked[1:-1, 1:-1])
            d = e
        if torch.equal(d, last):
            break
    cost = int(d[height, width])
    return INF if cost >= big else cost


def _best_value(w, v, cap):
    best = np.zeros(cap + 1, dtype=np.int64)
    for wi, vi in zip(w.tolist(), v.tolist()):
        if wi <= cap:
            best[wi:] = np.maximum(best[wi:], best[:cap + 1 - wi] + vi)
    return int(best[cap])
