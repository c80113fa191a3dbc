"""The step's default way of launching (launches, then a replayed graph on
small grids) against launches throughout: the same bits, through the step at
which the graph takes over, a marker count that changes, a switch of the
Poisson order and a rollback, with work on the null stream by another thread
meanwhile."""
import threading

import numpy as np
import pytest

from helpers import case, decomposition, gpu_for

pytestmark = pytest.mark.gpu


def test_default_launching_equals_launches():
    torch = pytest.importorskip("torch")
    c = case("cyl64")
    dec = decomposition(c)
    ge, gd = gpu_for(c, dec, axis="y"), gpu_for(c, dec, axis="y")
    ge.set_graph(False)
    stop, fail = threading.Event(), []

    def other():
        try:
            x = torch.ones(1024, device="cuda")
            while not stop.is_set():
                x = x * 0.5 + 0.5
                torch.cuda.current_stream().synchronize()
            assert float(x.sum()) == 1024.0
        except BaseException as e:   # noqa: B036
            fail.append(e)

    th = threading.Thread(target=other)
    th.start()
    try:
        t, dt = 0.0, c.params.dt0
        for ns in range(16):
            lmcc, lmvel, lmA = c.markers(t)
            if 8 <= ns < 12:
                lmcc, lmvel, lmA = lmcc[:20], lmvel[:20], lmA[:20]
            for g in (ge, gd):
                g.set_markers(np.asfortranarray(lmcc), np.asfortranarray(lmvel), np.ascontiguousarray(lmA))
                if ns == 6:
                    g.set_transform("z")
                if ns == 13:
                    g.save_state()
                    g.fluid_tsch(ns, 0.5 * dt, dt)
                    g.restore_state()
            dte, cfe = ge.fluid_tsch(ns, dt, dt)
            dtd, cfd = gd.fluid_tsch(ns, dt, dt)
            assert dte == dtd and cfe == cfd, ns
            se, sd = ge.get_state(), gd.get_state()
            for f in se:
                np.testing.assert_array_equal(se[f], sd[f], err_msg=f"{f} step {ns}")
            t += dte
            dt = dte
    finally:
        stop.set()
        th.join()
    assert not fail, fail
