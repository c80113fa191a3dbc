"""Tangents that carry over (k_loads_tau): markers whose probe is at rest take
the last tangent set before them, found within the wave, the workgroup of 256
markers or the workgroups before, and none before the first one that is set.

The velocity is zero in half of the domain or in stripes of it; there the
friction stress is the pressure's second derivatives times the carried
tangent, so it shows which marker's tangent was taken.  Bar as in the other
loads tests: 1e-9 of the largest value, against the oracle on the same
fields."""
import dataclasses

import numpy as np
import pytest

from helpers import case, decomposition, gpu_for, oracle_for, relmax, run_steps

pytestmark = pytest.mark.gpu


def _body(n):
    c = case("cyl64")
    th = -2.0 * np.pi * np.arange(n + 1) / n
    r = 0.5 * (c.verts[:, 0].max() - c.verts[:, 0].min())
    v = np.stack([c.center[0] + r * np.cos(th), c.center[1] + r * np.sin(th)], axis=1)
    v[-1] = v[0]
    return dataclasses.replace(c, verts=v, _rest=None)


@pytest.mark.parametrize("n", [63, 65, 256, 257, 1100])
@pytest.mark.parametrize("rest", ["second half", "first half", "stripes", "everywhere"])
def test_carried_tangents_match_the_oracle(n, rest):
    c = _body(n)
    dec = decomposition(c)
    o, g = oracle_for(c, dec), gpu_for(c, dec)
    run_steps(o, c, 1)
    run_steps(g, c, 1)
    st = g.get_state()
    rng = np.random.default_rng(n)
    z = np.concatenate([[c.zz[0]] * 3, 0.5 * (c.zz[:-1] + c.zz[1:]), [c.zz[-1]] * 3])
    k = np.arange(z.size)
    still = {"second half": z > c.center[1], "first half": z <= c.center[1], "stripes": (k // 6) % 2 == 0,
             "everywhere": z > -1.0}[rest]
    for f in ("q2", "q3", "pr"):
        st[f] = np.asfortranarray(rng.standard_normal(st[f].shape))
    for f in ("q2", "q3"):
        st[f][:, still] = 0.0
    g.set_state(st)
    o.set_state(st)
    nor, acc = c.surface(0.0)
    rc, po, to = o.loads_transfer(1.0, nor, acc)
    assert rc == 0
    pg, tg = g.loads_transfer(1.0, nor, acc)
    assert relmax(pg, po) <= 1e-9 and relmax(tg, to) <= 1e-9
    if rest != "everywhere":
        assert np.abs(to).max() > 0.0
    g.close()
