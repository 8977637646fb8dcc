"""Graphs that a caller captures of lbm_step on the grid's own stream: replayed
after other calls of an even number of steps in all -- odd calls in pairs, short
ones, a mask change with the steps that follow it, another variant, a tuning
call -- each replay is the steps it was captured of, bit for bit."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Graph:
    """lbm_step(g, n) captured on the grid's stream."""

    def __init__(self, g, n):
        from lbm_amd import _native as N
        self.hip, self.stream = N.load(), ctypes.c_void_p(g.stream)
        graph, self.exec = ctypes.c_void_p(), ctypes.c_void_p()
        assert self.hip.hipStreamBeginCapture(self.stream, 1) == 0
        g.step(n)
        assert self.hip.hipStreamEndCapture(self.stream, ctypes.byref(graph)) == 0
        assert self.hip.hipGraphInstantiate(ctypes.byref(self.exec), graph, None, None, ctypes.c_size_t(0)) == 0
        assert self.hip.hipGraphDestroy(graph) == 0

    def replay(self):
        assert self.hip.hipGraphLaunch(self.exec, self.stream) == 0

    def close(self):
        assert self.hip.hipGraphExecDestroy(self.exec) == 0


def _between(kind, g, mask):
    if kind == "odd calls":
        g.step(3)
        g.step(1)
    elif kind == "odd and short calls":
        g.step(5)
        g.step(2)
        g.step(9)
    elif kind == "mask":
        g.mask = mask
        g.step(2)  # the collision of the new state, then one step: a stream is pending
    elif kind == "long":
        g.step(50)
    elif kind == "variant":
        g.variant = 2
        g.step(4)
    elif kind == "tuned":
        g.autotune(4)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind", ["none", "odd calls", "odd and short calls", "mask", "long", "variant", "tuned"])
@pytest.mark.parametrize("n", [8, 20])
def test_replays(n, kind, precision):
    from lbm_amd import LBM, gen_circles
    print(f"case: caller's graph of {n} steps, {kind}, precision {precision}", flush=True)
    X, Y = 500, 130
    g, ref = (LBM(1.6, X, Y, precision=precision) for _ in range(2))
    ref.variant = 0
    for o in (g, ref):
        o.mask = gen_circles(X, Y, 3, 4, 5, 14)
        o.custom_speed(0.06)
        o.step(6)
    graph = Graph(g, n)  # (captured, not run)
    for again in range(3):
        graph.replay()
        ref.step(n)
        _between(kind, g, gen_circles(X, Y, 10 + again, 5, 5, 14))
        _between(kind if kind not in ("variant", "tuned") else "", ref, gen_circles(X, Y, 10 + again, 5, 5, 14))
        if kind == "variant":
            ref.step(4)
        graph.replay()
        ref.step(n)
        g.sync()
        for p, q in zip(g.moments(lagged=True), ref.moments(lagged=True)):
            assert np.array_equal(p, q), again
    assert np.array_equal(g.read_f().view(np.uint32), ref.read_f().view(np.uint32))
    graph.close()
    g.close()
    ref.close()
