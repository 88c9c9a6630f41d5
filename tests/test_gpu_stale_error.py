"""An error that an earlier HIP call of the calling thread left behind (the
caller's own, say) is not taken for one of this library's launches."""
import ctypes

import numpy as np
import pytest

import detectingscc_amd as scc
from oracle import pyoracle as orc
from helpers import assert_same_labels, random_graph

pytestmark = pytest.mark.gpu


def _leave_error():
    # refused by the runtime itself: there is no such device
    assert scc.lib().hipSetDevice(ctypes.c_int(1 << 20)) != 0


def test_calls_after_a_callers_error():
    rng = np.random.default_rng(3)
    gs = [random_graph(V, 3 * V, rng) for V in (5000, 80, 700)]
    _leave_error()
    with scc.Context(0) as ctx:
        for _ in range(2):   # the second upload is checked beside the graph that is there
            _leave_error()
            ctx.upload(gs[0])
            ctx.run(algo="g", sizes=False)
            assert_same_labels(ctx.labels(), orc.tarjan(gs[0])[0])
        _leave_error()
        ctx.batch_upload(scc.batch_from_graphs(gs))
        _leave_error()
        ctx.batch_run()
        _leave_error()
        labs, _ = ctx.batch_labels()
        for lab, g in zip(labs, gs):
            assert_same_labels(lab, orc.tarjan(g)[0])
