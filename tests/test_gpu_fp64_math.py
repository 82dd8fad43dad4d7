"""The FP64 kernels' own reciprocal (hardware estimate + two Newton steps) and
logarithm (atanh series after an exponent split), checked term by term: with
a single active source every output is one pair term, which numpy computes
from the same separation with its correctly rounded division and log.  The
sums' parity with the oracle is tested elsewhere; here each term must agree to
a few ulp, so a wrong coefficient or range reduction cannot hide inside a sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sphere_points(rng, n):
    p = rng.normal(size=(3, n))
    p /= np.linalg.norm(p, axis=0)
    return p


def _one_source(n_targets, rng):
    """Particle 0 is the only active source; particles 1.. are the targets."""
    p = _sphere_points(rng, n_targets + 1)
    act = np.zeros(n_targets + 1, np.int32)
    act[0] = 1
    area = np.zeros(n_targets + 1)
    area[0] = 0.37
    q = np.zeros(n_targets + 1)
    q[0] = 1.9
    return p, act, area, q


def _on_sphere_solver(ctx, p, q, area, act):
    """A device-resident FP64 solver with projected stages: its sums use the
    on-sphere form 1/2 |x - y|^2 of R^2 - x.y, with no R^2 - |x|^2 terms, so
    numpy can form the same denominator from the solver's positions."""
    from lpmgpu import BVESolver

    x, y, z = p
    s = BVESolver(ctx, x, y, z, q, area, act, absvort=2 * q, precision="fp64", project=True)
    st = s.state()
    pr, pa = s.stream()
    s.delete()
    return st, pr, pa


def test_fp64_log_in_sphere_green_sum(ctx):
    rng = np.random.default_rng(7)
    p, act, area, q = _one_source(20000, rng)
    # 200 targets within 1e-6 ... 1e-3 of the source, the rest anywhere
    near = p[:, :1] + rng.normal(size=(3, 200)) * np.geomspace(1e-6, 1e-3, 200)
    p[:, 1:201] = near / np.linalg.norm(near, axis=0)
    st, pr, pa = _on_sphere_solver(ctx, p, q, area, act)
    P = np.array([st["x"], st["y"], st["z"]])
    d = P[:, 1:] - P[:, :1]
    dd = 0.5 * np.sum(d * d, axis=0)  # R^2 - x.y in the kernel's form
    want = -np.log(dd) / (4 * np.pi) * q[0] * area[0]
    got = pr[1:]
    # |log| > 1: an ulp of difference in the squared distance (fma vs separate
    # products) moves log by 2e-16 absolute, below the tolerance only there
    big = np.abs(np.log(dd)) > 1.0
    rel = np.abs(got - want)[big] / np.abs(want)[big]
    assert rel.max() < 2e-15, rel.max()
    assert np.abs(got - want).max() < 4e-16 * np.abs(want).max()
    assert np.array_equal(pa[1:], 2 * pr[1:])


def test_fp64_log_in_plane_green_sum(ctx):
    rng = np.random.default_rng(8)
    n = 20000
    x = np.concatenate([[0.1], rng.uniform(-3, 3, n)])
    y = np.concatenate([[-0.2], rng.uniform(-3, 3, n)])
    # a few targets very close to the source and very far from it
    x[1:50] = 0.1 + rng.uniform(-1e-7, 1e-7, 49)
    y[1:50] = -0.2 + rng.uniform(-1e-7, 1e-7, 49)
    x[50:100] = 0.1 + rng.uniform(-1e4, 1e4, 50)
    act = np.zeros(n + 1, np.int32)
    act[0] = 1
    area = np.zeros(n + 1)
    area[0] = 0.5
    w = np.zeros(n + 1)
    w[0] = -1.3
    psi = ctx.plane_stream(x, y, w, area, act, precision="fp64")
    r2 = (x[1:] - x[0]) ** 2 + (y[1:] - y[0]) ** 2
    want = 0.5 * np.log(r2) / (2 * np.pi) * w[0] * area[0]
    big = np.abs(np.log(r2)) > 1.0
    rel = np.abs(psi[1:] - want)[big] / np.abs(want)[big]
    assert rel.max() < 2e-15, rel.max()


def test_fp64_reciprocal_in_biot_savart_sum(ctx):
    rng = np.random.default_rng(9)
    p, act, area, q = _one_source(20000, rng)
    near = p[:, :1] + rng.normal(size=(3, 200)) * np.geomspace(1e-6, 1e-3, 200)
    p[:, 1:201] = near / np.linalg.norm(near, axis=0)
    st, _, _ = _on_sphere_solver(ctx, p, q, area, act)
    P = np.array([st["x"], st["y"], st["z"]])
    # u_i = s (x_i - y) x x_i = s (x_i x y),  s = -zeta A / (4 pi (R^2 - x_i . y)),
    # R^2 - x.y = |x - y|^2 / 2; error scale |s| |x_i - y| (the size of each factor)
    d = P[:, 1:] - P[:, :1]
    den = 0.5 * np.sum(d * d, axis=0)
    s = -q[0] * area[0] / (4 * np.pi * den)
    want = np.cross(d.T, P[:, 1:].T).T * s
    got = np.array([st["u"][1:], st["v"][1:], st["w"][1:]])
    err = np.linalg.norm(got - want, axis=0) / (np.abs(s) * np.linalg.norm(d, axis=0))
    assert err.max() < 1e-14, err.max()


def test_fp64_exponential_in_pse_sums(ctx):
    """exp(-rho^2) of the 2nd-order kernel, one source term per target, from 0 to the
    smallest results.  rho^2 carries a relative rounding of a few ulp (coordinates
    scaled by 1 / eps, two differences and products), which the exponential turns into
    an error of rho^2 times that; below e^-700 the terms lose digits to denormals."""
    rng = np.random.default_rng(10)
    n = 20000
    eps = 0.25
    x = np.concatenate([[0.0], rng.uniform(-6.9, 6.9, n)])
    y = np.concatenate([[0.0], rng.uniform(-0.5, 0.5, n)])
    act = np.zeros(n + 1, np.int32)
    act[0] = 1
    area = np.zeros(n + 1)
    area[0] = 0.5
    f = np.zeros(n + 1)
    f[0] = 2.0
    lap = ctx.pse_plane_laplacian(x, y, f, area, act, eps, order=2, precision="fp64")[1:]
    q = (x[1:] / eps) ** 2 + (y[1:] / eps) ** 2
    want = 4 / np.pi / eps**4 * f[0] * area[0] * np.exp(-q)
    ok = q < 690
    rel = np.abs(lap - want)[ok] / want[ok]
    assert (rel < 2.3e-16 * (8 + 6 * q[ok])).all()
    far = q > 760
    assert far.any() and not lap[far].any()


@pytest.mark.parametrize("scale", [1e-100, 1e-60, 1e-30, 1.0, 1e30, 1e60, 1e70])
@pytest.mark.parametrize("n", [3, 64, 5000, 30011])
def test_fp64_reciprocals_in_fours(ctx, n, scale):
    """Four reciprocals from one of their product, taken one by one where the product
    leaves the range (separations from 1e38 on or below 1e-38).  Against numpy for 40
    targets: n terms of a few roundings each, 8 + sqrt(n) of 2^-53 of the terms' sum."""
    rng = np.random.default_rng(n)
    x, y = rng.uniform(-1, 1, n) * scale, rng.uniform(-1, 1, n) * scale
    w, area = rng.normal(size=n), np.full(n, scale / n)
    act = (rng.uniform(size=n) < 0.9).astype(np.int32)
    u, v = ctx.plane_velocity(x, y, w, area, act, precision="fp64")
    src = np.flatnonzero(act)
    for i in rng.integers(0, n, 40):
        j = src[src != i]
        dx, dy = (x[i] - x[j]) / scale, (y[i] - y[j]) / scale
        k = w[j] / n / (2 * np.pi * (dx * dx + dy * dy))
        tol = (8 + np.sqrt(n)) * 2.0**-53
        assert abs(u[i] + (k * dy).sum()) <= tol * np.abs(k * dy).sum()
        assert abs(v[i] - (k * dx).sum()) <= tol * np.abs(k * dx).sum()


def test_fp64_reciprocals_in_fours_keep_a_bad_value_to_its_target(ctx):
    """A passive particle on top of a source, and one that is not a number: NaN there,
    and every other target as without them."""
    n = 5000
    rng = np.random.default_rng(5)
    p = _sphere_points(rng, n)
    act = np.ones(n, np.int32)
    act[[70, 71]] = 0
    q, area = rng.normal(size=n), np.full(n, 4 * np.pi / n)
    ref = np.stack(ctx.bve_sphere_velocity(*p, q, area, act, precision="fp64"))
    p[:, 70] = p[:, 4000]
    p[0, 71] = np.nan
    got = np.stack(ctx.bve_sphere_velocity(*p, q, area, act, precision="fp64"))
    assert np.isnan(got[:, 71]).all() and not np.isfinite(got[:, 70]).any()
    rest = np.delete(np.arange(n), [70, 71])
    assert np.abs(got - ref)[:, rest].max() <= 1e-13 * np.abs(ref[:, rest]).max()
