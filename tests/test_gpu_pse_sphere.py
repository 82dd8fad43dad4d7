"""Sphere PSE Laplacian on the GPU (lpm_pse_sphere_laplacian) against the FP64
oracle (PSESphereLaplacianAtParticles, PSEDirectSum.f90:502-532) and the
reference's own spherePSETest thresholds."""
import numpy as np
import pytest

import lpmgpu
from helpers import icos

pytestmark = pytest.mark.gpu


def _harmonic(m):
    lat = np.arcsin(np.clip(m.z, -1, 1))
    lon = np.arctan2(m.y, m.x)
    return 3.0 * np.sqrt(35.0) * np.cos(4 * lon) * np.sin(lat) * (np.sin(lat) ** 2 - 1.0) ** 2


@pytest.mark.parametrize("level,eps", [(4, 0.3), (5, 0.05), (5, 0.12)])
def test_fp64_matches_oracle(ctx, oracle, level, eps):
    m = icos(level)
    f = _harmonic(m)
    ref = oracle.pse_sphere_laplacian(m.x, m.y, m.z, f, m.area, m.active, eps)
    got = ctx.pse_sphere_laplacian(m.x, m.y, m.z, f, m.area, m.active, eps, precision="fp64")
    e = np.abs(got - ref).max() / np.abs(ref).max()
    print(f"L{level} eps {eps}: fp64 vs oracle {e:.2e}")
    assert e < 1e-11


@pytest.mark.parametrize("level,eps", [(5, 0.05), (5, 0.12), (4, 0.3)])
def test_fp32_matches_oracle(ctx, oracle, level, eps):
    """eps = 0.05 takes the series form of the distance (7 eps <= 0.56 R), the
    others the asin form."""
    m = icos(level)
    f = _harmonic(m)
    ref = oracle.pse_sphere_laplacian(m.x, m.y, m.z, f, m.area, m.active, eps)
    got = ctx.pse_sphere_laplacian(m.x, m.y, m.z, f, m.area, m.active, eps, precision="fp32")
    e = np.abs(got - ref).max() / np.abs(ref).max()
    print(f"L{level} eps {eps}: fp32 vs oracle {e:.2e}")
    assert e < 1e-4


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_reference_regression_thresholds(ctx, precision):
    """spherePSETest (tests/CMakeLists.txt:74-75): icosahedral nest 3, eps = h^0.6,
    L_inf <= 0.0175 over all particles and squared L2 <= 1.18e-4 over rank 0's
    block of 4 (SpherePSEConvTest.f90:314-316, 374-389) for a Laplacian -30 f."""
    m = icos(3)
    f = _harmonic(m)
    eps = lpmgpu.pse_eps(m.max_edge_length, 0.6)
    lap = ctx.pse_sphere_laplacian(m.x, m.y, m.z, f, m.area, m.active, eps, precision=precision)
    exact = -30.0 * f
    err = np.abs(lap - exact)
    linf = float(err.max() / np.abs(exact).max())
    s, e, _ = lpmgpu.load_balance(m.n, 4)
    blk = np.zeros(m.n, bool)
    blk[s[0] - 1: e[0]] = True
    act = (m.active == 1) & blk
    l2 = float((err[act] ** 2 * m.area[act]).sum() / (exact[act] ** 2 * m.area[act]).sum())
    print(precision, "linf", linf, "l2", l2)
    assert linf <= 0.0175 and l2 <= 1.18e-4


def test_blocks_concatenate(ctx):
    """Target blocks concatenate to the full call (the source split count follows
    the block size, so FP64 agrees to rounding, not bitwise)."""
    m = icos(4)
    f = _harmonic(m)
    full = ctx.pse_sphere_laplacian(m.x, m.y, m.z, f, m.area, m.active, 0.2, precision="fp64")
    parts = np.zeros(m.n)
    for i0, i1 in ((0, 1000), (1000, 5000), (5000, m.n)):
        got = ctx.pse_sphere_laplacian(m.x, m.y, m.z, f, m.area, m.active, 0.2, i0=i0, i1=i1, precision="fp64")
        assert np.all(got[:i0] == 0.0) and np.all(got[i1:] == 0.0)
        parts[i0:i1] = got[i0:i1]
    assert np.abs(parts - full).max() < 1e-13 * np.abs(full).max()


def test_bad_arguments(ctx):
    m = icos(2)
    f = _harmonic(m)
    with pytest.raises(lpmgpu.LpmError):
        ctx.pse_sphere_laplacian(m.x, m.y, m.z, f, m.area, m.active, -1.0)
    with pytest.raises(lpmgpu.LpmError):
        ctx.pse_sphere_laplacian(m.x, m.y, m.z, f, m.area, m.active, 0.1, radius=0.0)
    # the context survives
    ctx.pse_sphere_laplacian(m.x, m.y, m.z, f, m.area, m.active, 0.3)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("reach", [0.345, 0.355, 0.555, 0.565, 0.695, 0.705, 1.155, 1.165, 1.195, 1.205])
def test_distance_series_at_the_ends_of_their_ranges(ctx, oracle, precision, reach):
    """Each series of the great-circle distance on both sides of the largest 7 eps / R
    it is used for (FP64 0.35, 0.70, 1.16; FP32 0.56, 1.2), on a radius other than 1,
    against the oracle's asin form: the bars of the sums above."""
    radius = 3.0
    m = icos(4)
    x, y, z, area = m.x * radius, m.y * radius, m.z * radius, m.area * radius**2
    f = _harmonic(m)
    eps = reach / 7.0 * radius
    ref = oracle.pse_sphere_laplacian(x, y, z, f, area, m.active, eps, radius=radius)
    got = ctx.pse_sphere_laplacian(x, y, z, f, area, m.active, eps, radius=radius, precision=precision)
    e = np.abs(got - ref).max() / np.abs(ref).max()
    assert e < (1e-11 if precision == "fp64" else 1e-4), e
