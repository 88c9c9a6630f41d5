"""The single-graph engine's one-launch path for small graphs: on both sides
of its size limits and of the size up to which a graph is held in LDS whole,
against Tarjan, with the counts it reports."""
import numpy as np
import pytest

import detectingscc_amd as scc
from oracle import pyoracle as orc
from helpers import assert_same_labels, random_graph

pytestmark = pytest.mark.gpu

# (V, arcs): the LDS limit is 8 (V + 2) + 2 E = 36,864 words, the path's
# limits are 16,384 vertices and 2^18 arcs
SIZES = ((1, 0), (1, 3), (2, 5), (64, 200), (1000, 14424), (1000, 14425), (2302, 5), (4606, 0), (4607, 9000),
         (4096, 1 << 18), (4096, (1 << 18) + 1), (16383, 40000), (16384, 70000), (16385, 70000))


@pytest.mark.parametrize("algo,t1,t2", [("g", True, True), ("x", False, False), ("h", True, True), ("y", False, False)])
def test_small_graphs(algo, t1, t2):
    rng = np.random.default_rng(11)
    with scc.Context(0) as ctx:
        for V, E in SIZES:
            g = random_graph(V, E, rng)
            want, n = orc.tarjan(g)
            ctx.upload(g)
            for _ in range(2):
                st = ctx.run(algo=algo, trim1=t1, trim2=t2, sizes=False)
                what = f"V={V} E={E} -a {algo} trims {t1:d}{t2:d}"
                assert_same_labels(ctx.labels(), want, what)
                assert st.num_sccs == n, what
                assert st.largest == 0 and st.ms_scc > 0, what
                # every SCC is found by a trim or by a pivot, trim-2's in pairs
                assert st.num_trim1 + st.num_trim2 + st.num_pivot == n, what
            # the sizes pass and the device-wide engine agree on the same graph
            sized = ctx.run(algo=algo, trim1=t1, trim2=t2, sizes=True)
            assert sized.num_sccs == n, what
            hist = dict(ctx.histogram()[0])
            sizes = np.bincount(want[1:].astype(np.int64), minlength=V + 1)
            assert hist == {int(k): int(c) for k, c in zip(*np.unique(sizes[sizes > 0], return_counts=True))}, what
