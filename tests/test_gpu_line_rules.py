"""Line solves where their launch rules change, and one line or column to the
other side.

The Helmholtz j-lines take four waves per workgroup up to 512 planes and eight
above, in as many workgroups as take every line at once (up to 1024 planes); a
batch takes eight and as many lines per wave as keep its workgroups resident.
Every line is solved by one wave with the same operations whatever the shape,
so an instance alone and the same instance in a batch (on the transform tiles
of the instance alone) give the same bits.

The one-pass k-lines with chunks of 9 to 16 rows own eight columns per
workgroup up to 1024 columns and sixteen above; every form does the operations
of the three passes in the same order."""
import numpy as np
import pytest

from fribois2d_amd import cases
from helpers import gpu_for

pytestmark = pytest.mark.gpu


def _case(n2m, n3m):
    h = 0.02
    rc, zz = np.linspace(0.0, n2m * h, n2m + 1), np.linspace(0.0, n3m * h, n3m + 1)
    p = cases.FluidParams(n2=n2m + 1, n3=n3m + 1, alx3=n3m * h, rext2=n2m * h, visc=0.01, dt0=1.0e-4, ibact=False)
    return cases.Case(f"rules{n2m}x{n3m}", p, rc, zz, None, (0.5 * n2m * h, 0.5 * n3m * h), None, 20261205)


# 512 | 513 planes: four | eight waves; 1024 | 1025: one | two rounds of them;
# 17, 49: one line more than whole workgroups hold
@pytest.mark.parametrize("n2m,n3m", [(20, 17), (20, 49), (30, 512), (30, 513), (30, 1024), (30, 1025)])
def test_j_lines_where_the_rule_changes(n2m, n3m):
    from fribois2d_amd.gpu import FluidBatch
    c = _case(n2m, n3m)
    alone, member, other = gpu_for(c), gpu_for(c), gpu_for(_case(24, 40))
    b = FluidBatch([member, other])
    b.set_gemm_shape(0)
    dt = np.full(2, c.params.dt0)
    for ns in range(2):
        dta, _ = alone.fluid_tsch(ns, dt[0], dt[0])
        dt = b.step(ns, dt)[0]
        assert dt[0] == dta
    sa, sm = alone.get_state(), member.get_state()
    for f in sa:
        assert np.isfinite(sa[f]).all() and np.array_equal(sa[f], sm[f]), f
    b.close()


@pytest.mark.parametrize("n2m,n3m", [(1024, 513), (1025, 513), (1040, 1024), (1041, 600)])
def test_k_lines_where_the_rule_changes(n2m, n3m):
    st = []
    for form in ("fused", "3pass"):
        g = gpu_for(_case(n2m, n3m))
        g.set_ksolve(form)
        dt = g.params.dt0
        for ns in range(2):
            dt, _ = g.fluid_tsch(ns, dt, dt)
        st.append(g.get_state())
        g.close()
    for f in st[0]:
        assert np.isfinite(st[0][f]).all() and np.array_equal(st[0][f], st[1][f]), f


def _alone_and_together(sizes, axis):
    """Fields of the instances after two steps alone and after two steps as a
    batch on 32x32 transform tiles."""
    from fribois2d_amd.gpu import FluidBatch
    cs = [_case(*s) for s in sizes]
    gs, out = [gpu_for(c, axis=axis) for c in cs], []
    b = FluidBatch(gs)
    b.set_gemm_shape(0)
    dt = np.array([c.params.dt0 for c in cs])
    for ns in range(2):
        dt, _, err = b.step(ns, dt)
        assert not err.any()
    together = [g.get_state() for g in gs]
    b.close()
    for i, c in enumerate(cs):
        gs[i].close()
        a, d = gpu_for(c, axis=axis), c.params.dt0
        for ns in range(2):
            d, _ = a.fluid_tsch(ns, d, d)
        assert d == dt[i]
        out.append((a.get_state(), together[i]))
        a.close()
    return out


# Pressure partials of a batch's taller tiles (kb_upd): the large members make
# the tiles eight planes tall, the others' partials cover 1, 2 and 4 of them,
# the last tiles are cut short (z order: the first member has no y order);
# then four planes with partials of one in the mirror form, 160 and 61 planes
@pytest.mark.parametrize("sizes,axis", [
    ([(70, 63), (620, 1100), (620, 1101), (311, 517), (311, 700), (64, 97)], "z"),
    ([(126, 160)] * 26 + [(50, 61), (63, 97), (64, 130)], "y"),
])
def test_batch_pressure_partials_are_those_of_the_instances_alone(sizes, axis):
    for i, (alone, together) in enumerate(_alone_and_together(sizes, axis)):
        for f in alone:
            assert np.isfinite(alone[f]).all() and np.array_equal(alone[f], together[f]), (sizes[i], f)
