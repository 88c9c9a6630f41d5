"""detectSCC's search across the partitions: when it runs, where it is given
up, and the labels in each case."""
import re

import numpy as np
import pytest

import detectingscc_amd as scc
from oracle import pyoracle as orc
from helpers import assert_same_labels

pytestmark = pytest.mark.gpu


def _grid(side, rng, p=0.8, diagonals=False):
    x = np.arange(side * side).reshape(side, side) + 1
    s, d = [], []
    pairs = [(x[:, :-1], x[:, 1:]), (x[:, 1:], x[:, :-1]), (x[:-1], x[1:]), (x[1:], x[:-1])]
    if diagonals:   # more than four arcs per vertex and direction
        pairs += [(x[:-1, :-1], x[1:, 1:]), (x[1:, 1:], x[:-1, :-1])]
    for a, b in pairs:
        keep = rng.random(a.shape) < p
        s.append(a[keep])
        d.append(b[keep])
    return scc.from_arcs(side * side, np.concatenate(s), np.concatenate(d))


def _communities(k, size, between, rng):
    """k random graphs of `size` vertices and 6 arcs each, and `between` arcs
    from each to the next (the last to the first)."""
    V = k * size
    s = rng.integers(0, V, 6 * V)
    d = s // size * size + rng.integers(0, size, s.size)
    c = np.repeat(np.arange(k), between)
    s = np.concatenate([s, c * size + rng.integers(0, size, c.size)])
    d = np.concatenate([d, (c + 1) % k * size + rng.integers(0, size, c.size)])
    return scc.from_arcs(V, s + 1, d + 1)


def _part(V, p):
    part = np.zeros(V + 2, np.uint32)
    part[1:V + 1] = p
    return part


def _run(g, parts, **kw):
    want, n = orc.tarjan(g)
    with scc.Context(0) as ctx:
        ctx.upload(g)
        for part in parts:
            ctx.upload_partition(_part(g.V, part))
            for trims in (True, False):
                for sizes in (False, True):
                    st = ctx.run(algo="d", trim1=trims, trim2=trims, sizes=sizes)
                    assert_same_labels(ctx.labels(), want, f"trims {trims} sizes {sizes}")
                    assert st.num_sccs == n


@pytest.mark.parametrize("between", [0, 1, 40, 2000])
@pytest.mark.parametrize("k,size", [(2, 40), (12, 3000), (60, 1500)])
def test_communities(k, size, between):
    """Partitions without, with few and with many arcs between them."""
    g = _communities(k, size, between, np.random.default_rng(between + k))
    _run(g, [np.arange(g.V) // size])


@pytest.mark.parametrize("side,diagonals", [(150, False), (700, False), (100, True), (900, True)])
def test_high_diameter(side, diagonals):
    """Low-degree graphs, which are searched to the end, and others, whose
    search ends within the bound, is given up, or is given the longer one."""
    rng = np.random.default_rng(side)
    g = _grid(side, rng, 0.6 if diagonals else 0.8, diagonals)
    _run(g, [np.arange(g.V) * 16 // g.V, rng.integers(0, 16, g.V)])


def test_search_keeps_its_bound(monkeypatch, capfd):
    """On a grid with diagonals in blocks of rows no level past the sixteenth
    is run."""
    g = _grid(1200, np.random.default_rng(1), p=0.6, diagonals=True)
    monkeypatch.setenv("SCC_TRACE_LEVELS", "1")
    with scc.Context(0) as ctx:
        ctx.upload(g)
        ctx.upload_partition(_part(g.V, np.arange(g.V) * 16 // g.V))
        capfd.readouterr()
        ctx.run(algo="d", sizes=False)
    looks = [int(x) for x in re.findall(r"\[scc reach\] after level (\d+):", capfd.readouterr().err)]
    first = [looks[0]]
    for x in looks[1:]:
        if x < first[-1]:
            break
        first.append(x)
    assert first[-1] == 15, first
