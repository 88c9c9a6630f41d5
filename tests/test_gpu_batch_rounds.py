"""The batched kernel's first round and list phases at the sizes and shapes
where they change path: graphs at the edges of a chunk (64 vertices) and of
the LDS tiers, with hubs walked by the whole workgroup, sparse enough to be
trimmed and searched top-down only, dense enough for bottom-up levels, and
with thousands of SCCs that the first round leaves to the list phases."""
import threading

import numpy as np
import pytest
import torch

import detectingscc_amd as scc
from oracle import pyoracle as orc
from helpers import assert_same_labels, random_graph

pytestmark = pytest.mark.gpu

EDGES = (1, 2, 63, 64, 65, 127, 129, 2047, 2050, 4097, 8193, 65535, 65536, 65537)


def _islands(V, rng):
    """Disjoint cycles of 1 to 9 vertices over permuted ids, joined by arcs
    from an island to a random later one: every cycle is an SCC."""
    perm = rng.permutation(V) + 1
    cuts = np.unique(np.concatenate([[0, V], np.cumsum(rng.integers(1, 10, V))]))
    cuts = cuts[cuts <= V]
    src, dst = [], []
    for a, b in zip(cuts[:-1], cuts[1:]):
        ring = perm[a:b]
        if ring.size > 1:
            src.append(ring)
            dst.append(np.roll(ring, -1))
    k = V // 4
    a, b = rng.integers(0, V, k), rng.integers(0, V, k)
    island = np.searchsorted(cuts, np.arange(V), side="right")
    keep = island[a] < island[b]
    src.append(perm[a[keep]])
    dst.append(perm[b[keep]])
    return scc.from_arcs(V, np.concatenate(src), np.concatenate(dst))


def _hubs(V, rng):
    """A third of the arcs leave, and a third enter, one of three vertices."""
    E = 6 * V
    src, dst = rng.integers(1, V + 1, E), rng.integers(1, V + 1, E)
    src[:E // 3] = rng.integers(1, min(V, 3) + 1, E // 3)
    dst[E // 3:2 * E // 3] = rng.integers(1, min(V, 3) + 1, E // 3)
    return scc.from_arcs(V, src, dst)


@pytest.mark.parametrize("block", [256, 512, 1024])
@pytest.mark.parametrize("shape", ["islands", "hubs", "sparse", "dense"])
def test_batch_first_round_and_lists(shape, block):
    rng = np.random.default_rng([block, len(shape)])
    make = {"islands": _islands, "hubs": _hubs, "sparse": lambda V, r: random_graph(V, 2 * V, r),
            "dense": lambda V, r: random_graph(V, 9 * V, r)}[shape]
    gs = [make(V, rng) for V in EDGES]
    want = [orc.tarjan(g) for g in gs]
    with scc.Context(0) as ctx:
        ctx.batch_upload(scc.batch_from_graphs(gs))
        for algo, t1, t2 in (("g", True, True), ("g", False, False), ("h", True, False), ("h", False, False)):
            ctx.batch_run(algo=algo, trim1=t1, trim2=t2, lanes=16, block=block)
            labs, nscc = ctx.batch_labels()
            for i, (lab, n) in enumerate(want):
                what = f"{shape} V={EDGES[i]} -a {algo} trims {t1:d}{t2:d} block {block}"
                assert_same_labels(labs[i], lab, what)
                assert nscc[i] == n, what


@pytest.mark.parametrize("slack", [0, 7, 5000])
def test_batch_labels_layout(slack):
    """Labels land at the host layout's offsets whatever the distance between
    two graphs' rows (one copy, or graph by graph where the gaps are wide),
    and the words between them stay the caller's."""
    rng = np.random.default_rng(slack)
    gs = [random_graph(V, 3 * V, rng) for V in (1, 70, 2, 333, 64, 1000, 63)]
    b = scc.batch_from_graphs(gs)
    row = np.zeros(len(gs) + 1, np.uint64)
    row[1:] = np.cumsum([g.V + 2 + slack for g in gs])
    row += np.uint64(slack)
    Fr, Br = np.zeros(int(row[-1]), np.uint32), np.zeros(int(row[-1]), np.uint32)
    for i, g in enumerate(gs):
        Fr[int(row[i]):int(row[i]) + g.V + 2] = g.Fr
        Br[int(row[i]):int(row[i]) + g.V + 2] = g.Br
    b = scc.Batch(b.V, b.E, row, b.col_off, Fr, b.Fc, Br, b.Bc)
    lab = np.full(int(row[-1]), 0xABCD, np.uint32)
    own = np.zeros(lab.size, bool)
    with scc.Context(0) as ctx:
        ctx.batch_upload(b)
        ctx.batch_run()
        assert scc.lib().scc_batch_labels(ctx._ctx, scc._p32(lab), None) == 0
    for i, g in enumerate(gs):
        at = int(row[i])
        own[at:at + g.V + 1] = True
        assert_same_labels(lab[at:at + g.V + 1], orc.tarjan(g)[0], f"slack {slack} graph {i}")
    assert (lab[~own] == 0xABCD).all()


@pytest.mark.parametrize("starts", [(0, 204, 102, 306), (102, 0, 204, 306), (204, 102, 0, 306), (7, 1000, 500, 5000),
                                    (5000, 0, 9000, 200)])
def test_batch_labels_row_order(starts):
    """Rows in any order: graph i's rows, and its labels, are at row_off[i]."""
    rng = np.random.default_rng(sum(starts))
    gs = [random_graph(100, 300, rng) for _ in range(len(starts))]
    n = max(starts) + 102
    row = np.array(starts + (starts[-1] + 102,), np.uint64)
    Fr, Br = np.zeros(n, np.uint32), np.zeros(n, np.uint32)
    for at, g in zip(starts, gs):
        Fr[at:at + 102], Br[at:at + 102] = g.Fr, g.Br
    b = scc.batch_from_graphs(gs)
    b = scc.Batch(b.V, b.E, row, b.col_off, Fr, b.Fc, Br, b.Bc)
    lab = np.full(n, 0xABCD, np.uint32)
    nscc = np.zeros(len(gs), np.uint32)
    with scc.Context(0) as ctx:
        ctx.batch_upload(b)
        ctx.batch_run()
        assert scc.lib().scc_batch_labels(ctx._ctx, scc._p32(lab), scc._p32(nscc)) == 0
    for i, (at, g) in enumerate(zip(starts, gs)):
        want, k = orc.tarjan(g)
        assert_same_labels(lab[at:at + 101], want, f"rows at {starts}, graph {i}")
        assert nscc[i] == k
        lab[at:at + 101] = 0xABCD
    assert (lab == 0xABCD).all()


@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("spacing", [0, 61])
def test_batch_labels_gaps_stay_the_callers(pinned, spacing):
    """A word between two graphs' labels that another thread counts in while
    the labels are copied loses no count, in pageable and page-locked memory."""
    rng = np.random.default_rng(spacing)
    gs = [random_graph(V, 2 * V, rng) for V in rng.integers(1, 6000, 700)]
    b = scc.batch_from_graphs(gs)
    row = np.zeros(len(gs) + 1, np.uint64)
    row[1:] = np.cumsum([g.V + 2 + spacing for g in gs])
    Fr, Br = np.zeros(int(row[-1]), np.uint32), np.zeros(int(row[-1]), np.uint32)
    for at, g in zip(row.astype(int), gs):
        Fr[at:at + g.V + 2], Br[at:at + g.V + 2] = g.Fr, g.Br
    b = scc.Batch(b.V, b.E, row, b.col_off, Fr, b.Fc, Br, b.Bc)
    lab = torch.full((int(row[-1]),), 0xABCD, dtype=torch.int32, pin_memory=pinned).numpy().view(np.uint32)
    mine = int(row[len(gs) // 2]) + gs[len(gs) // 2].V + 1
    lab[mine] = 0
    counted, stop = 0, threading.Event()

    def count():
        nonlocal counted
        while not stop.is_set():
            lab[mine] += 1
            counted += 1

    with scc.Context(0) as ctx:
        ctx.batch_upload(b)
        ctx.batch_run()
        t = threading.Thread(target=count)
        t.start()
        status = [scc.lib().scc_batch_labels(ctx._ctx, scc._p32(lab), None) for _ in range(20)]
        stop.set()
        t.join()
    assert status == [0] * 20 and counted > 0
    assert int(lab[mine]) == counted & 0xFFFFFFFF
    lab[mine] = 0xABCD
    for i, (at, g) in enumerate(zip(row.astype(int), gs)):
        assert_same_labels(lab[at:at + g.V + 1], orc.tarjan(g)[0], f"graph {i}")
        lab[at:at + g.V + 1] = 0xABCD
    assert (lab == 0xABCD).all()
