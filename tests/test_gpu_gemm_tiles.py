"""The transform GEMM at the edges of its tiles (fribo_gemm.hip: 32x32, 32x64
and 96x128 tiles, K-slices of 32 and 24 with remainders, operands with and
without the 16-byte alignment of the direct-to-LDS loads) and the mirror form
with halves of every remainder.

Bar of a product: each element is a sum of K products, so its error is at
most K * 2^-53 * (|A| |B|) to first order; twice that is allowed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# last: five 32x64 units against twelve of 96x128 and six of 32x32; twelve
# 96x128 units against as many of the smaller tiles
SIZES = [(1, 1, 1), (2, 3, 4), (31, 33, 31), (32, 32, 32), (33, 31, 33), (64, 65, 63), (95, 129, 25), (97, 127, 96),
         (143, 181, 145), (1064, 1300, 40), (1536, 2048, 49)]


@pytest.mark.parametrize("form", ["nt", "nn"])
@pytest.mark.parametrize("pad", [16, 0])
@pytest.mark.parametrize("size", SIZES)
def test_products_at_tile_edges(form, pad, size):
    from fribois2d_amd import gpu
    M, N, K = size
    rng = np.random.default_rng([M, N, K])
    A = rng.standard_normal((M, K))
    B = rng.standard_normal((N, K) if form == "nt" else (K, N))
    C = (gpu.gemm_nt if form == "nt" else gpu.gemm_nn)(A, B, pad=pad)
    Bk = B.T if form == "nt" else B
    assert (np.abs(C - A @ Bk) <= 2.0 * K * 2.0 ** -53 * (np.abs(A) @ np.abs(Bk))).all()


@pytest.mark.parametrize("n2m", [10, 64, 94, 130, 190, 262])
def test_mirror_form_projects(n2m):
    """Halves of 5, 32, 47, 65, 95 and 131 rows: each tile row holds rows of
    one half only, and the second half starts on an odd row.  A step ends
    divergence-free: what is left is the rounding of the velocities over the
    spacing (2^-53 / 0.02 = 6e-15) and of the Poisson solve (its condition
    number, 1e5 here, times 2^-53 of the 0.05 the perturbation brings), both
    below 1e-12; a wrong row of the transforms would leave 1e-3 or more."""
    from fribois2d_amd import cases
    from fribois2d_amd.gpu import FluidStep
    n3m = n2m + 37
    rc, zz = np.linspace(0.0, 6.0, n2m + 1), np.linspace(0.0, 8.0, n3m + 1)
    p = cases.FluidParams(n2=n2m + 1, n3=n3m + 1, alx3=8.0, rext2=6.0, visc=0.02, ibact=False)
    g = FluidStep(p, rc, zz)
    assert g.transform == "y" and g.ymirror
    g.set_state(cases.initial_state(p, 9))
    g.fluid_tsch(0, p.dt0)
    assert g.diagnostics()["divmax"] <= 1e-10
    g.close()


@pytest.mark.parametrize("n3m", [6, 127, 129, 512, 513, 1024, 1025, 2048, 2049])
@pytest.mark.parametrize("n2m", [5, 14])
def test_mode_lines_project(n3m, n2m):
    """The per-mode z-lines at the edges of their chunk classes (chunks of 2
    to 8, 9 to 16 and 17 to 32 rows in one pass, longer ones in three).  A
    step ends divergence-free to rounding: the condition number of the Poisson
    operator times 2^-53 of the divergence the step starts from, and 2^-53
    over the spacing; 16 times that is allowed."""
    from fribois2d_amd import cases
    from fribois2d_amd.gpu import FluidStep
    rc, zz = np.linspace(0.0, 6.0, n2m + 1), np.linspace(0.0, 8.0, n3m + 1)
    p = cases.FluidParams(n2=n2m + 1, n3=n3m + 1, alx3=8.0, rext2=6.0, visc=0.02, ibact=False)
    g = FluidStep(p, rc, zz)
    assert g.transform == ("y" if n2m < n3m else "z")
    g.set_state(cases.initial_state(p, 9))
    div0 = g.diagnostics()["divmax"]
    g.fluid_tsch(0, p.dt0)
    hy, hz = 6.0 / n2m, 8.0 / n3m
    kappa = (4.0 / hy ** 2 + 4.0 / hz ** 2) / (np.pi / 8.0) ** 2
    assert g.diagnostics()["divmax"] <= 16.0 * 2.0 ** -53 * (kappa * div0 + 1.0 / min(hy, hz))
    g.close()
