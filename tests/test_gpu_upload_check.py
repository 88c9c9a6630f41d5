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


@pytest.mark.parametrize("graphs,vmax,degree", [(1, 1, 0), (1, 70000, 3), (9, 600, 4), (300, 200, 5), (9000, 12, 2)])
def test_batch_faults_are_refused(graphs, vmax, degree):
    rng = np.random.default_rng(graphs)
    sizes = [vmax] * graphs if graphs == 1 else rng.integers(1, vmax + 1, graphs)
    good = scc.batch_from_graphs([random_graph(int(v), int(v) * degree, rng) for v in sizes])
    wants = [orc.tarjan(good.graph(i)) for i in range(0, graphs, max(1, graphs // 50))]
    with scc.Context(0) as ctx:
        for g in sorted({0, graphs // 2, graphs - 1}):
            V, E = int(good.V[g]), int(good.E[g])
            faults = [("Fr", "row_off", v, E + 1) for v in {2, V} if V >= 2]
            faults += [("Br", "row_off", v, E + 1) for v in {2, V} if V >= 2]
            faults += [(a, "col_off", k, c) for a in ("Fc", "Bc") if E for k in {0, E // 2, E - 1}
                       for c in (0, V + 1, 0xFFFFFFFF)]
            for name, off, at, value in faults:
                arrays = {k: getattr(good, k).copy() for k in ("Fr", "Fc", "Br", "Bc")}
                arrays[name][int(getattr(good, off)[g]) + at] = value
                bad = scc.Batch(good.V, good.E, good.row_off, good.col_off, arrays["Fr"], arrays["Fc"],
                                arrays["Br"], arrays["Bc"])
                with pytest.raises(scc.SCCError, match="invalid CSR"):
                    ctx.batch_upload(bad)
                with pytest.raises(scc.SCCError, match="no batch"):
                    ctx.batch_run()
        ctx.batch_upload(good)
        ctx.batch_run()
        labels, counts = ctx.batch_labels()
        for k, i in enumerate(range(0, graphs, max(1, graphs // 50))):
            assert counts[i] == wants[k][1]
            assert_same_labels(labels[i], wants[k][0], f"graph {i}")


@pytest.mark.parametrize("graphs", [1, 3, 12])
def test_faults_in_small_batches(graphs):
    """Batches small enough for the host's check, on both sides of its limit."""
    rng = np.random.default_rng(graphs)
    for degree in (3, 40):   # up to 12 graphs of 38 to 60 vertices, then more than 2^15 words
        good = scc.batch_from_graphs([random_graph(int(v), int(v) * degree, rng) for v in rng.integers(38, 61, graphs)])
        with scc.Context(0) as ctx:
            for g in (0, graphs - 1):
                V, E = int(good.V[g]), int(good.E[g])
                for name, off, at, value in (("Fr", "row_off", 2, E + 1), ("Br", "row_off", V, E + 1),
                                             ("Fc", "col_off", 0, 0), ("Fc", "col_off", E - 1, V + 1),
                                             ("Bc", "col_off", 0, V + 1), ("Bc", "col_off", E - 1, 0xFFFFFFFF)):
                    arrays = {k: getattr(good, k).copy() for k in ("Fr", "Fc", "Br", "Bc")}
                    arrays[name][int(getattr(good, off)[g]) + at] = value
                    with pytest.raises(scc.SCCError, match="invalid CSR"):
                        ctx.batch_upload(scc.Batch(good.V, good.E, good.row_off, good.col_off, arrays["Fr"],
                                                   arrays["Fc"], arrays["Br"], arrays["Bc"]))
                    with pytest.raises(scc.SCCError, match="no batch"):
                        ctx.batch_run()
            ctx.batch_upload(good)
            ctx.batch_run()
            for i, lab in enumerate(ctx.batch_labels()[0]):
                assert_same_labels(lab, orc.tarjan(good.graph(i))[0], f"graph {i}")


def test_batch_of_wrong_offsets_is_none():
    """A larger batch whose offsets are refused does not run in the buffers of
    the batch before."""
    rng = np.random.default_rng(8)
    good = scc.batch_from_graphs([random_graph(9, 20, rng) for _ in range(3)])
    more = scc.batch_from_graphs([random_graph(50, 200, rng) for _ in range(500)])
    col = more.col_off.copy()
    col[-1] += 1
    wrong = scc.Batch(more.V, more.E, more.row_off, col, more.Fr, more.Fc, more.Br, more.Bc)
    with scc.Context(0) as ctx:
        ctx.batch_upload(good)
        ctx.batch_run()
        with pytest.raises(scc.SCCError, match="offsets do not match"):
            ctx.batch_upload(wrong)
        for call in (ctx.batch_run, ctx.batch_run_serial, ctx.batch_autotune):
            with pytest.raises(scc.SCCError, match="no batch uploaded"):
                call()
        ctx.batch_upload(more)
        ctx.batch_run()
        assert_same_labels(ctx.batch_labels()[0][499], orc.tarjan(more.graph(499))[0])
