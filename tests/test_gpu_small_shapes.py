"""The one-launch path for small graphs on structured graphs: cycles, grids,
chains and islands of small SCCs, vertices with more arcs than a wave walks
for one lane, for graphs held whole in LDS and for larger ones, against
Tarjan; and its time on the last of these."""
import time

import numpy as np
import pytest

import detectingscc_amd as scc
from oracle import pyoracle as orc
from helpers import assert_same_labels

pytestmark = pytest.mark.gpu


def _cycle(V, rng):
    a = np.arange(1, V + 1)
    return V, [a], [np.roll(a, -1)]


def _grid(V, rng):
    side = int(V ** 0.5)
    x = np.arange(side * side).reshape(side, side) + 1
    s, d = [], []
    for a, b in ((x[:, :-1], x[:, 1:]), (x[:, 1:], x[:, :-1]), (x[:-1], x[1:]), (x[1:], x[:-1])):
        keep = rng.random(a.shape) < 0.7
        s.append(a[keep])
        d.append(b[keep])
    return side * side, s, d


def _islands(V, rng):
    """Rings of three; half lead to one vertex, which leads to the others."""
    k = (V - 1) // 3
    ring = np.arange(1, 3 * k + 1).reshape(k, 3)
    hub = np.full(k, 3 * k + 1)
    return (3 * k + 1, [ring, ring[:k // 2, 0], hub[k // 2:]],
            [np.roll(ring, -1, axis=1), hub[:k // 2], ring[k // 2:, 0]])


def _star(V, rng):
    """No cycle: sources to one vertex, which leads to the sinks."""
    k = V // 2
    return V, [np.arange(2, k), np.full(V - k, 1)], [np.full(k - 2, 1), np.arange(k + 1, V + 1)]


def _pairs(V, rng):
    """A clique, a vertex behind it that leads to a chain of 2-cycles."""
    k = 40
    n = (V - k - 1) // 2 * 2
    a = np.arange(k + 2, k + 2 + n, 2)
    x, y = np.meshgrid(np.arange(1, k + 1), np.arange(1, k + 1))
    return (k + 1 + n, [x, [1], np.full(n, k + 1), a, a + 1, a[:-1] + 1],
            [y, [k + 1], np.arange(k + 2, k + 2 + n), a + 1, a, a[1:]])


def _path(V, rng):
    """Two random SCCs of V/8 vertices at the ends of a path, every vertex of
    which also leads to one vertex before the second."""
    k = V // 8
    hub = V
    mid = np.arange(k, V - 1 - k)
    s = [np.arange(1, k + 1), np.full(k - 1, 1), np.arange(2, k + 1), mid, np.full(mid.size, 0) + mid, [hub],
         np.arange(V - k, V), rng.integers(V - k, V, 4 * k)]
    d = [np.r_[np.arange(2, k + 1), 1], np.arange(2, k + 1), np.full(k - 1, 1), mid + 1, np.full(mid.size, hub),
         [V - k], np.r_[np.arange(V - k + 1, V), V - k], rng.integers(V - k, V, 4 * k)]
    return V, s, d


def _graph(make, V):
    rng = np.random.default_rng(V)
    V, s, d = make(V, rng)
    ids = rng.permutation(V) + 1
    flat = lambda x: ids[np.concatenate([np.asarray(y).ravel() for y in x]).astype(np.int64) - 1]
    return scc.from_arcs(V, flat(s), flat(d))


@pytest.mark.parametrize("V", [1200, 1700, 5000, 16384])
@pytest.mark.parametrize("make", [_cycle, _grid, _islands, _star, _pairs, _path])
def test_small_shapes(make, V):
    g = _graph(make, V)
    want, n = orc.tarjan(g)
    deep = make in (_pairs, _path) and V > 1700   # colouring takes long there, as in the reference
    with scc.Context(0) as ctx:
        ctx.upload(g)
        for algo, t1, t2 in (("g", True, True), ("x", False, False), ("h", True, True), ("y", False, False)):
            if deep and algo in "hy" and make is _path:
                continue
            st = ctx.run(algo=algo, trim1=t1, trim2=t2, sizes=False)
            what = f"{make.__name__} V={V} -a {algo} trims {t1:d}{t2:d}"
            assert_same_labels(ctx.labels(), want, what)
            assert st.num_sccs == n, what
            assert st.num_trim1 + st.num_trim2 + st.num_pivot == n, what


def test_long_rows_do_not_hold_a_lane():
    """A vertex with 4,000 out-arcs whose row every colour pass folds: in one
    launch at most a third of the device-wide engine's time."""
    g = _graph(_pairs, 4096)
    ms = {}
    with scc.Context(0) as ctx:
        ctx.upload(g)
        for wide in (False, True):
            best = 1e9
            for _ in range(4):
                t0 = time.perf_counter()
                ctx.run(algo="h", sizes=False, phase_times=wide)
                best = min(best, time.perf_counter() - t0)
            ms[wide] = best * 1e3
    assert ms[False] * 3 < ms[True], ms


def test_parallel_arcs():
    """A chain whose every arc is there 1,000 times, all of which trim-1 peels
    vertex by vertex: no slower in one launch than device-wide."""
    V, k = 200, 1000
    a = np.repeat(np.arange(1, V), k)
    ids = np.random.default_rng(5).permutation(V) + 1
    g = scc.from_arcs(V, ids[a - 1], ids[a])
    ms = {}
    with scc.Context(0) as ctx:
        ctx.upload(g)
        for wide in (False, True):
            best = 1e9
            for _ in range(4):
                t0 = time.perf_counter()
                st = ctx.run(algo="g", sizes=False, phase_times=wide)
                best = min(best, time.perf_counter() - t0)
                assert_same_labels(ctx.labels(), np.arange(V + 1, dtype=np.uint32))
                assert st.num_sccs == V
            ms[wide] = best * 1e3
    print(ms)
    assert ms[False] < ms[True], ms


def _trimmed(g, once):
    """Live vertices after trim-1: one pass, or the fixpoint."""
    src = np.repeat(np.arange(g.V + 1), np.diff(g.Fr.astype(np.int64)))
    dst = g.Fc.astype(np.int64)
    live = np.arange(g.V + 1) > 0
    while True:
        ok = live[src] & live[dst]
        keep = live & (np.bincount(src[ok], minlength=g.V + 1) > 0) & (np.bincount(dst[ok], minlength=g.V + 1) > 0)
        if once or (keep == live).all():
            return keep
        live = keep


def _hub_dag(V, rng):
    """A random SCC and a vertex of many arcs that only trim-1's second pass
    removes: sources to it, it to sinks."""
    k = V // 20
    body = V - 2 * k - 1
    hub = body + 1
    ring = np.arange(1, body + 1)
    return V, [ring, rng.integers(1, body + 1, 4 * body), np.arange(hub + 1, hub + 1 + k), np.full(k, hub), [hub]], [
        np.roll(ring, -1), rng.integers(1, body + 1, 4 * body), np.full(k, hub), np.arange(hub + 1 + k, V + 1), [1]]


@pytest.mark.parametrize("V", [900, 1700, 4000, 16384])
@pytest.mark.parametrize("arcs", ["hub", 2, 4, 8])
def test_small_counts(V, arcs):
    """What is trimmed, and the pivot elected from the rest: trim-1 to its
    fixpoint under Hong's order, one pass of it before colouring."""
    g = _graph(_hub_dag, V) if arcs == "hub" else scc.gen_er(V, arcs * V, 4, 2, 64, seed=V)
    _, n = orc.tarjan(g)
    Fr, Br = g.Fr.astype(np.int64), g.Br.astype(np.int64)
    product = np.minimum(np.diff(Fr) * np.diff(Br), 0xFFFFFFFF)
    with scc.Context(0) as ctx:
        ctx.upload(g)
        for algo in "gxhy":
            st = ctx.run(algo=algo, trim1=True, trim2=False, sizes=False)
            live = _trimmed(g, once=algo in "hy")
            first = int(np.argmax(np.where(live, product, -1)))
            assert st.first_pivot == first, f"-a {algo}"
            if algo in "hy":
                assert st.num_trim1 == g.V - live.sum()
            elif arcs == "hub":
                assert (st.num_trim1, st.num_pivot) == (n - 1, 1)
            else:
                assert st.num_trim1 >= g.V - live.sum()
