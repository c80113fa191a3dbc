"""State transfer: what is set comes back bit for bit, whole and in windows,
below one staging chunk, over several and past the ring (fribo_xfer.hip:
chunks of 524288 doubles, three of them in flight)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FIELDS = ("q2", "q3", "pr", "ru2", "ru3")


def _step(n3m, n2m):
    from fribois2d_amd import cases
    from fribois2d_amd.gpu import FluidStep
    rc, zz = np.linspace(0.0, 6.0, n2m + 1), np.linspace(0.0, 8.0, n3m + 1)
    p = cases.FluidParams(n2=n2m + 1, n3=n3m + 1, alx3=8.0, rext2=6.0, visc=0.02, ibact=False)
    return p, FluidStep(p, rc, zz)


# total doubles of the state: 204; 68k; 1.4M (three chunks); 3.3M (seven)
@pytest.mark.parametrize("n3m,n2m", [(4, 4), (131, 97), (560, 499), (900, 720)])
def test_state_round_trip(n3m, n2m):
    p, g = _step(n3m, n2m)
    rng = np.random.default_rng(n3m)
    st = {k: np.asfortranarray(rng.standard_normal((n2m + 1, n3m + 6))) for k in ("q2", "q3", "pr")}
    st.update({k: np.asfortranarray(rng.standard_normal((n2m + 1, n3m))) for k in ("ru2", "ru3")})
    st.update({k: rng.standard_normal(n2m + 1) for k in ("qb2s", "qb3s", "qb2n", "qb3n", "dq2x2o", "dq3x2o")})
    for _ in range(2):
        g.set_state(st)
        back = g.get_state()
        for k in st:
            assert np.array_equal(back[k], st[k]), k
    # a window that starts in the ghost planes, one plane, and the last planes
    for a, b in ((-2, 1), (n3m // 2, n3m // 2), (n3m - 1, n3m + 3)):
        win = {k: np.full_like(st[k], np.nan) for k in FIELDS}
        g.fetch_fields(a, b, win, FIELDS)
        for k in FIELDS:
            base, last = (1, n3m) if k.startswith("ru") else (-2, n3m + 3)
            lo, hi = max(a, base) - base, min(b, last) - base + 1
            assert np.array_equal(win[k][:, lo:hi], st[k][:, lo:hi]), (k, a, b)
            assert np.isnan(win[k][:, :lo]).all() and np.isnan(win[k][:, hi:]).all(), (k, a, b)
    # part of the state: the rest stays
    g.set_state({"q3": st["q2"]})
    back = g.get_state()
    assert np.array_equal(back["q3"], st["q2"]) and np.array_equal(back["q2"], st["q2"])
    g.close()


def test_pressure_means_of_a_read_back():
    """After a step the whole read-back and the windows agree on the pressure,
    whose pending means differ between the interior and the outer entries."""
    from fribois2d_amd import cases
    p, g = _step(131, 97)
    g.set_state(cases.initial_state(p, 3))
    dt, _ = g.fluid_tsch(0, p.dt0)
    g.fluid_tsch(1, dt)
    st = g.get_state()
    win = {"pr": np.full_like(st["pr"], np.nan)}
    for a in range(-2, 131 + 4, 7):
        g.fetch_fields(a, min(a + 6, 131 + 3), win, ("pr",))
    assert np.array_equal(win["pr"], st["pr"])
    area = np.outer(np.diff(np.linspace(0.0, 6.0, 98)), np.diff(np.linspace(0.0, 8.0, 132)))
    assert abs((st["pr"][:97, 3:134] * area).sum()) <= 1e-12 * np.abs(st["pr"]).max() * area.sum()
    g.close()
