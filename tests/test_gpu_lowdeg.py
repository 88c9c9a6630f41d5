"""High-diameter searches on graphs of at most four arcs per vertex and
direction, which run from rows of their own, and on graphs just past that."""
import numpy as np
import pytest

import detectingscc_amd as scc
from oracle import pyoracle as orc
from helpers import assert_same_labels

pytestmark = pytest.mark.gpu


def _cycle(V, arcs, rng):
    """A cycle through all vertices; vertex 1 and its neighbours get `arcs`
    out- and in-arcs in all."""
    a = np.arange(1, V + 1)
    s, d = [a], [np.roll(a, -1)]
    for k in range(2, arcs + 1):
        s += [[1], [1 + k]]
        d += [[1 + k], [1]]
    return V, s, d


def _grid(V, side, rng):
    x = np.arange(side * side).reshape(side, side) + 1
    s, d = [], []
    for a, b in ((x[:, :-1], x[:, 1:]), (x[:, 1:], x[:, :-1]), (x[:-1], x[1:]), (x[1:], x[:-1])):
        keep = rng.random(a.shape) < 0.8
        s.append(a[keep])
        d.append(b[keep])
    return side * side, s, d


def _burst(V, arcs, rng):
    """A long path into a random graph of `arcs` permutations (a frontier that
    grows from one vertex to most of them) and a long path back."""
    n = V // 2
    body = np.arange(n) + 1
    s = [body] * arcs
    d = [rng.permutation(n) + 1 for _ in range(arcs)]
    path = np.arange(n + 1, V + 1)
    s.append(path)
    d.append(np.append(path[1:], 1))
    s.append([n])
    d.append([n + 1])
    return V, s, d


@pytest.mark.parametrize("make,V,par", [(_cycle, 20000, 1), (_cycle, 20000, 4), (_cycle, 20000, 5), (_grid, 0, 160),
                                        (_grid, 0, 300), (_burst, 40000, 2), (_burst, 120000, 3), (_burst, 40000, 4)])
@pytest.mark.parametrize("trims", [True, False])
def test_low_degree(make, V, par, trims):
    rng = np.random.default_rng(V + par)
    V, s, d = make(V, par, rng)
    ids = rng.permutation(V) + 1
    g = scc.from_arcs(V, ids[np.concatenate(s).astype(np.int64) - 1], ids[np.concatenate(d).astype(np.int64) - 1])
    want, n = orc.tarjan(g)
    with scc.Context(0) as ctx:
        ctx.upload(g)
        for sizes in (False, True, False):
            st = ctx.run(algo="g", trim1=trims, trim2=trims, sizes=sizes)
            what = f"{make.__name__} {V} {par} trims {trims} sizes {sizes}"
            assert_same_labels(ctx.labels(), want, what)
            assert st.num_sccs == n, what
