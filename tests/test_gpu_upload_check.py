"""Uploads the device checks (and, below their size, the host): every fault a
row or column array can have is refused, and the graph held before stays."""
import numpy as np
import pytest

import detectingscc_amd as scc
from oracle import pyoracle as orc
from helpers import assert_same_labels, random_graph

pytestmark = pytest.mark.gpu


def _faults(V, E):
    """(array, index, value) of single faults, with the message's end."""
    for rows, cols in (("Fr", "Fc"), ("Br", "Bc")):
        yield rows, 0, 1, "row array must start 0,0"
        yield rows, 1, 1, "row array must start 0,0"
        yield rows, V + 1, E - 1, "row array must start 0,0"
        for v in (2, V // 2, V):
            yield rows, v, E + 1, "row array is not monotone"
        for k in (0, E // 2, E - 1):
            for c in (0, V + 1, 0xFFFFFFFF):
                yield cols, k, c, "column entry outside"


@pytest.mark.parametrize("V,E", [(50, 4000), (4095, 4095), (4096, 900), (300, 4096), (30000, 100003)])
@pytest.mark.parametrize("held", ["none", "larger", "smaller"])
def test_faults_are_refused(V, E, held):
    rng = np.random.default_rng(V + E)
    g = random_graph(V, E, rng)
    want, n = orc.tarjan(g)
    old = {"none": None, "larger": random_graph(40000, 130000, rng), "smaller": random_graph(20, 30, rng)}[held]
    with scc.Context(0) as ctx:
        if old is not None:
            ctx.upload(old)
            old_want, old_n = orc.tarjan(old)
        for name, at, value, message in _faults(g.V, g.E):
            arrays = {k: np.array(getattr(g, k), np.uint32) for k in ("Fr", "Fc", "Br", "Bc")}
            arrays[name][at] = value
            bad = scc.Graph(g.V, g.E, arrays["Fr"], arrays["Fc"], arrays["Br"], arrays["Bc"])
            with pytest.raises(scc.SCCError, match=f"{name[0]}r/{name[0]}c {message}"):
                ctx.upload(bad)
        if old is not None:
            assert ctx.run().num_sccs == old_n
            assert_same_labels(ctx.labels(), old_want, "the graph held before")
        for _ in range(2):
            ctx.upload(g)
            assert ctx.run().num_sccs == n
            assert_same_labels(ctx.labels(), want, "after the refusals")
