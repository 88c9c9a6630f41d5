"""Arrays an engine can do without (the second set of graph arrays, the
low-degree rows) are given back where an allocation fails."""
import numpy as np
import pytest

import detectingscc_amd as scc
from oracle import pyoracle as orc
from helpers import assert_same_labels

pytestmark = pytest.mark.gpu


def _rings(V, rng):
    """Rings of eight over permuted ids, each joined to a later one."""
    ids = rng.permutation(V).reshape(-1, 8) + 1
    k = ids.shape[0]
    a = np.arange(k - 1)
    b = a + 1 + rng.integers(0, k - 1 - a)
    return scc.from_arcs(V, np.concatenate([ids.ravel(), ids[a, 0]]),
                         np.concatenate([np.roll(ids, -1, axis=1).ravel(), ids[b, 1]]))


def _detect(g, part, uploads, want):
    with scc.Context(0) as ctx:
        for _ in range(uploads):   # from the second on there are two sets of graph arrays
            ctx.upload(g)
        ctx.run(algo="g", sizes=False)   # a graph of at most two arcs per vertex
        ctx.upload_partition(part)
        ctx.run(algo="d", sizes=False)
        assert_same_labels(ctx.labels(), want, f"{uploads} uploads")


def test_optional_arrays_are_given_back(monkeypatch):
    rng = np.random.default_rng(2)
    g = _rings(40000, rng)
    want, _ = orc.tarjan(g)
    part = np.zeros(g.V + 2, np.uint32)
    part[1:g.V + 1] = rng.integers(0, 2, g.V)
    second_set = 8 * (g.V + 2 + g.E)
    # the least scratch memory with which one upload's run goes through
    for limit in range(second_set, 64 * second_set, second_set // 4):
        monkeypatch.setenv("SCC_SCRATCH_LIMIT", str(limit))
        try:
            _detect(g, part, 1, want)
            break
        except scc.SCCError as e:
            assert e.status == 4
    # the second set fits it too, and must not be what the run then lacks
    _detect(g, part, 2, want)
    _detect(g, part, 3, want)
