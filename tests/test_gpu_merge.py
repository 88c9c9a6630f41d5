"""detectSCC: its search for the SCC across the partitions, and the local SCCs
and quotient graph of what that leaves or of everything."""
import numpy as np
import pytest

import detectingscc_amd as scc
from oracle import pyoracle as orc
from helpers import assert_same_labels

pytestmark = pytest.mark.gpu


def _rings(k, size, joined, rng):
    """k rings of `size` vertices over permuted ids; the first `joined` of
    them on one cycle of rings (one SCC), the next ones too as a second such
    cycle of two, the others joined to later rings only."""
    V = k * size
    ids = rng.permutation(V).reshape(k, size) + 1
    src, dst = [ids.ravel()], [np.roll(ids, -1, axis=1).ravel()]
    order = np.arange(joined)
    src.append(ids[order, 0])
    dst.append(ids[np.roll(order, -1), 0])
    if k >= joined + 2:
        src.append(ids[[joined, joined + 1], 1])
        dst.append(ids[[joined + 1, joined], 1])
    a = rng.integers(0, k, 3 * k)
    b = rng.integers(0, k, 3 * k)
    keep = (a < b) & (a >= joined)
    src.append(ids[a[keep], 0])
    dst.append(ids[b[keep], size - 1])
    return scc.from_arcs(V, np.concatenate(src), np.concatenate(dst))


@pytest.mark.parametrize("k,size,joined", [(1, 40, 1), (300, 7, 300), (300, 7, 120), (300, 33, 0), (9, 31, 2),
                                           (4000, 5, 3900)])
@pytest.mark.parametrize("trims", [True, False])
def test_merge_shapes(k, size, joined, trims):
    """All in one SCC, most, none, and a long cycle of rings (a search that
    is given up); partitions that split the rings and that join them."""
    rng = np.random.default_rng(k + size)
    g = _rings(k, size, joined, rng)
    want, n = orc.tarjan(g)
    with scc.Context(0) as ctx:
        ctx.upload(g)
        for parts in (1, 3, 50):
            part = np.zeros(g.V + 2, np.uint32)
            part[1:g.V + 1] = rng.integers(0, parts, g.V)
            ctx.upload_partition(part)
            for sizes in (False, True):
                st = ctx.run(algo="d", trim1=trims, trim2=trims, sizes=sizes)
                what = f"{k} rings of {size}, {joined} joined, {parts} partitions, trims {trims}, sizes {sizes}"
                assert_same_labels(ctx.labels(), want, what)
                assert st.num_sccs == n, what
