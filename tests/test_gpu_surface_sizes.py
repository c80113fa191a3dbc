"""Loads, forcing check and diagnostics at the marker counts and grid extents
where their kernels split the work differently: fewer markers than a wave, a
wave and one more, more than the workgroup of the forcing check; a marker on
the inflow plane (not inside the domain, so without loads); grids with fewer
and more cells than the diagnostics' threads and blocks.

Bars as in test_gpu_loads: 1e-9 of the maximum for the loads after steps of
the fluid; the norms of the forcing check are the binary tree over 1024
partial sums, reproduced here operation by operation, so they are equal;
extrema equal, tree sums to 1e-13.
"""
import dataclasses

import numpy as np
import pytest

from helpers import case, decomposition, gpu_for, oracle_for, relmax, run_steps

pytestmark = pytest.mark.gpu


def body(n):
    c = case("cyl64")
    th = -2.0 * np.pi * np.arange(n + 1) / n
    r = 0.5 * (c.verts[:, 0].max() - c.verts[:, 0].min())
    v = np.stack([c.center[0] + r * np.cos(th), c.center[1] + r * np.sin(th)], axis=1)
    v[-1] = v[0]
    return dataclasses.replace(c, verts=v, _rest=None)


class Moved:
    """Solver whose marker ``i`` is put on the inflow plane z = 0."""

    def __init__(self, s, i):
        self.s, self.i = s, i

    def set_markers(self, cc, vel, a):
        cc = cc.copy(order="F")
        cc[self.i, 1] = 0.0
        self.s.set_markers(cc, vel, a)

    def fluid_tsch(self, *a):
        return self.s.fluid_tsch(*a)


def tree_norm(err):
    s = np.zeros(1024)
    for i in range(0, err.size, 1024):
        e = err[i:i + 1024]
        s[:e.size] += e * e
    while s.size > 1:
        s = s[:s.size // 2] + s[s.size // 2:]
    return np.sqrt(s[0]) / err.size


@pytest.mark.parametrize("n", [7, 64, 65, 1025])
def test_loads_and_forcing_check_at_any_marker_count(n):
    c = body(n)
    dec = decomposition(c)
    o, g = oracle_for(c, dec), gpu_for(c, dec)
    run_steps(Moved(o, n // 2), c, 2)
    run_steps(Moved(g, n // 2), c, 2)
    nor, acc = c.surface(0.0)
    rc, po, to = o.loads_transfer(1.0, nor, acc)
    assert rc == 0
    pg, tg = g.loads_transfer(1.0, nor, acc)
    assert pg[n // 2] == 0.0 and np.all(tg[n // 2] == 0.0)
    assert relmax(pg, po) <= 1e-9 and relmax(tg, to) <= 1e-9
    bv, bw, nv, nw = g.checkbcs()
    assert nv == tree_norm(bv) and nw == tree_norm(bw)
    assert bv[n // 2] == 0.0 and bw[n // 2] == 0.0


@pytest.mark.parametrize("n2m,n3m", [(8, 8), (257, 40), (40, 300)])
def test_diagnostics_at_any_extent(n2m, n3m):
    c = case("cyl64")
    p = dataclasses.replace(c.params, n2=n2m + 1, n3=n3m + 1, alx3=20.0, ibact=0)
    c = dataclasses.replace(c, params=p, rc=np.linspace(0.0, p.rext2, n2m + 1), zz=np.linspace(0.0, p.alx3, n3m + 1),
                            verts=None, _rest=None)
    dec = decomposition(c)
    o, g = oracle_for(c, dec), gpu_for(c, dec)
    rng = np.random.default_rng(n2m)
    st = g.get_state()
    for k in ("q2", "q3", "pr"):
        st[k] = np.asfortranarray(rng.standard_normal(st[k].shape))
    g.set_state(st)
    o.set_state({k: st[k] for k in ("q2", "q3", "pr")})
    do, dg = o.diagnostics(), g.diagnostics()
    for k in ("vmax2", "vmax3", "vmin2", "vmin3", "divmax", "cflm"):
        assert dg[k] == do[k], k
    # sums of n2m * n3m terms of order one times the cell's area
    for k in ("ektot", "q3avg", "vorti"):
        assert abs(dg[k] - do[k]) <= 1e-13 * max(abs(do[k]), 1.0), k


def test_restored_state_repeats_the_step():
    """Save, step, restore, step: the same bits."""
    c = case("cyl64")
    g = gpu_for(c)
    _, dt = run_steps(g, c, 2)
    g.save_state()
    run_steps(g, c, 1, dt=dt, t0=0.3, ns0=2)
    a = g.get_state()
    run_steps(g, c, 2, dt=dt, t0=0.5, ns0=3)
    g.restore_state()
    run_steps(g, c, 1, dt=dt, t0=0.3, ns0=2)
    b = g.get_state()
    for k in a:
        assert np.array_equal(a[k], b[k]), k
