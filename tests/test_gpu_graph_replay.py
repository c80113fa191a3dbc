"""Which steps replay a graph where the caller has not said: on small grids
those from the third with the same marker buffers on, and none on large ones
or after set_graph(False); with set_graph(True) every one.  The same while
another thread works on the null stream, which must not break off the
capture."""
import threading

import numpy as np
import pytest

from fribois2d_amd import cases
from helpers import case, decomposition, gpu_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def torch_first():
    """torch before the library, so that both use one HIP runtime (torch finds
    no device after the library has loaded another)."""
    return pytest.importorskip("torch")


def _steps(g, c, n, ns0=0, nlm=None):
    out, dt = [], c.params.dt0
    for ns in range(ns0, ns0 + n):
        lm = c.markers(0.0)
        g.set_markers(*(np.asfortranarray(x[:nlm]) for x in lm))
        g.fluid_tsch(ns, dt, dt)
        out.append(g.replayed)
    return out


def _run(c):
    g = gpu_for(c, decomposition(c))
    assert g.replayed is None
    assert _steps(g, c, 5) == [False, False, True, True, True]
    assert _steps(g, c, 4, 5, nlm=20) == [False, False, True, True]
    g.set_transform("z")
    assert _steps(g, c, 1, 9, nlm=20) == [True]
    g.set_graph(False)
    assert _steps(g, c, 2, 10, nlm=20) == [False, False]
    g.set_graph(True)
    assert _steps(g, c, 2, 12) == [True, True]
    g.close()


def test_default_steps_replay_from_the_third_on():
    _run(case("cyl64"))


def test_the_null_stream_of_another_thread_does_not_stop_the_capture(torch_first):
    torch = torch_first
    stop, ready, fail = threading.Event(), threading.Event(), []

    def other():
        try:
            x = torch.ones(1024, device="cuda")
            while not stop.is_set():
                x = x * 0.5 + 0.5
                torch.cuda.current_stream().synchronize()
                ready.set()
        except BaseException as e:   # noqa: B036
            fail.append(e)

    th = threading.Thread(target=other)
    th.start()
    try:
        assert ready.wait(60), fail
        for _ in range(3):
            _run(case("cyl64"))
    finally:
        stop.set()
        th.join()
    assert not fail, fail


# 299 712 | 300 608 cells (the rule's line: 300 000)
@pytest.mark.parametrize("n3m,expect", [(669, True), (671, False)])
def test_only_small_grids_replay_by_default(n3m, expect):
    n2m = 448
    h = 0.02
    p = cases.FluidParams(n2=n2m + 1, n3=n3m + 1, alx3=n3m * h, rext2=n2m * h, visc=0.01, dt0=1.0e-4, ibact=False)
    c = cases.Case("line", p, np.linspace(0.0, n2m * h, n2m + 1), np.linspace(0.0, n3m * h, n3m + 1), None, None, None, 7)
    g = gpu_for(c)
    seen = []
    for ns in range(4):
        g.fluid_tsch(ns, p.dt0, p.dt0)
        seen.append(g.replayed)
    g.close()
    assert seen == [False, False, expect, expect]
