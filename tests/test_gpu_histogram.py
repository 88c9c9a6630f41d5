"""Size histograms of 1 to 300 different SCC sizes (the count and the first
255 pairs come back in one copy, any others in a second one), and of sizes
that occur often."""
import numpy as np
import pytest

import detectingscc_amd as scc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kinds", [1, 2, 254, 255, 256, 257, 300])
@pytest.mark.parametrize("sizes", [True, False])
def test_many_sizes(kinds, sizes):
    rng = np.random.default_rng(kinds)
    each = np.concatenate([np.arange(1, kinds + 1), np.minimum(np.arange(3000) % 7 + 1, kinds)])
    V = int(each.sum())
    ids = rng.permutation(V) + 1
    start = np.concatenate([[0], np.cumsum(each)])[:-1]
    owner = np.repeat(np.arange(each.size), each)
    at = np.arange(V)
    nxt = np.where(at + 1 < start[owner] + each[owner], at + 1, start[owner])
    g = scc.from_arcs(V, ids[at], ids[nxt])
    with scc.Context(0) as ctx:
        ctx.upload(g)
        st = ctx.run(sizes=sizes)
        assert st.num_sccs == each.size
        want = {int(k): int(c) for k, c in zip(*np.unique(each, return_counts=True))}
        for _ in range(2):
            assert dict(ctx.histogram()[0]) == want
