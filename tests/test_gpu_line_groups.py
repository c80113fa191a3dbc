"""Line solves at the edges of their launch rules.

The one-pass k-lines own 4, 8 or 16 columns per workgroup by the grid's width
and chunk length; every form does the operations of the three passes in the
same order, so the step's results are the same bits.  The j-lines run four or
eight waves per workgroup by the number of lines: on both sides of that line
the step agrees with the oracle to 1e-10 of the field maximum after two steps
(the multi-step bar)."""
import numpy as np
import pytest

from fribois2d_amd import cases
from helpers import decomposition, gpu_for, oracle_for, relmax, run_steps

pytestmark = pytest.mark.gpu


def _case(n2m, n3m):
    h = 0.02
    rc, zz = np.linspace(0.0, n2m * h, n2m + 1), np.linspace(0.0, n3m * h, n3m + 1)
    p = cases.FluidParams(n2=n2m + 1, n3=n3m + 1, alx3=n3m * h, rext2=n2m * h, visc=0.01, dt0=1.0e-4)
    yc, zc = 0.5 * n2m * h, 0.5 * n3m * h
    verts = cases.cylinder_vertices(yc, zc, 0.06, 24)
    return cases.Case(f"lines{n2m}x{n3m}", p, rc, zz, verts, (yc, zc), None, 20261205)


# (512 | 513, 512) chunks of 8 rows, four | eight columns; (n, 513) and (n,
# 1024) chunks of 9 and 16; (1024 | 1025, 1025) chunks of 17, eight | sixteen
@pytest.mark.parametrize("n2m,n3m", [(9, 16), (512, 512), (513, 512), (43, 513), (30, 1024), (1024, 1025), (1025, 1025)])
def test_one_pass_k_lines_equal_the_three_passes(n2m, n3m):
    c = _case(n2m, n3m)
    c = cases.Case(c.name, c.params, c.rc, c.zz, None, c.center, None, c.seed)
    st = []
    for form in ("fused", "3pass"):
        g = gpu_for(c)
        g.set_ksolve(form)
        run_steps(g, c, 2)
        st.append(g.get_state())
    for f in st[0]:
        assert np.array_equal(st[0][f], st[1][f]), f


@pytest.mark.parametrize("n3m", [768, 769])
def test_j_lines_on_both_sides_of_the_wave_rule(n3m):
    c = _case(70, n3m)
    dec = decomposition(c)
    o, g = oracle_for(c, dec), gpu_for(c, dec)
    run_steps(o, c, 2)
    run_steps(g, c, 2)
    so, sg = {k: o.get(k) for k in ("q2", "q3", "pr")}, g.get_state()
    for f in ("q2", "q3", "pr"):
        e = relmax(sg[f], so[f])
        print(f"n3m={n3m} {f}: {e:.2e}", flush=True)
        assert e <= 1e-10, f
