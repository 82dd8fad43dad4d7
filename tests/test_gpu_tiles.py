"""The tile paths of large sums: spatial order, far tiles on the MFMA.

Each call is compared with the all-pairs kernel (a forced tile shape) and with the
FP64 sum of the same inputs, over input orders, ragged blocks and masks, sizes at
the edges of tiles, and values that are not finite.  FP32 velocity and stream sums
are held to 1e-6 of the largest value, the library's FP32 bar on meshes."""
import numpy as np
import pytest

from helpers import rel_err_max
from lpmgpu import BVEBatch, BVESolver, _lib as L
from lpmgpu import ic, mesh

pytestmark = pytest.mark.gpu

TOL32 = 1e-6


def _rows(out):
    return [out] if isinstance(out, np.ndarray) else [np.asarray(o) for o in out]


def _all_pairs(ctx, kind, prec, call):
    ctx.set_tuning(kind, prec, 2, 256 if prec == "fp32" else 64, 0)
    try:
        return _rows(call())
    finally:
        ctx.set_tuning(kind, prec, 0, 0, 0)


def _sphere(order, seed=3):
    """Icosahedral level 6 (122,882 particles), turned, in the mesh's order or shuffled."""
    m = mesh.icosahedral_mesh(6)
    rng = np.random.default_rng(seed)
    rot, _ = np.linalg.qr(rng.normal(size=(3, 3)))
    xyz = m.xyz() @ rot
    idx = rng.permutation(m.n) if order == "shuffled" else np.arange(m.n)
    x, y, z = (np.ascontiguousarray(c[idx]) for c in xyz.T)
    zeta = ic.random_gaussian_vortices(rng, 3, x, y, z) + ic.rh4_vorticity(x, y, z)
    active = m.active[idx] * (rng.uniform(size=m.n) < 0.8)
    return x, y, z, zeta, m.area[idx], active.astype(np.int32)


@pytest.mark.parametrize("order", ["mesh", "shuffled"])
@pytest.mark.parametrize("block", [(0, None), (17, 122882 - 255), (5, 5 + 256 * 128 + 1)])
def test_far_tiles_sphere(ctx, order, block):
    x, y, z, zeta, area, act = _sphere(order)
    i0, i1 = block[0], block[1] or x.size
    for kind, call in (
            (L.K_SPHERE_BS, lambda p: ctx.bve_sphere_velocity(x, y, z, zeta, area, act, i0=i0, i1=i1, precision=p)),
            (L.K_SPHERE_GREEN, lambda p: ctx.bve_sphere_stream(x, y, z, zeta, zeta + z, area, act, i0=i0, i1=i1,
                                                               precision=p))):
        got, ref = _rows(call("fp32")), _rows(call("fp64"))
        for g, r in zip(got, ref):
            assert rel_err_max(g[i0:i1], r[i0:i1]) < TOL32
            assert not g[:i0].any() and not g[i1:].any()
        for g, r in zip(got, _all_pairs(ctx, kind, "fp32", lambda: call("fp32"))):
            assert rel_err_max(g, r) < 2 * TOL32
        again = _rows(call("fp32"))
        assert all(np.array_equal(a, b) for a, b in zip(got, again))


@pytest.mark.parametrize("shape", ["grid", "strip", "two_clusters", "duplicates"])
def test_far_tiles_plane(ctx, shape):
    """Layouts that make balls large, thin, far apart or of radius zero."""
    rng = np.random.default_rng(7)
    n = 70000
    if shape == "grid":
        x, y, area, _ = mesh.grid_centres(270, 1.0, jitter=5e-4, seed=2)
    elif shape == "strip":
        x, y = rng.uniform(-50, 50, n), rng.uniform(-0.01, 0.01, n)
    elif shape == "two_clusters":
        x, y = rng.normal(size=n) * 0.1, rng.normal(size=n) * 0.1
        x[::2] += 40.0
    else:  # every point 300 times over: the pairs of equal points are self-like, with weight 0
        x, y = np.repeat(rng.uniform(-1, 1, n // 300), 300), np.repeat(rng.uniform(-1, 1, n // 300), 300)
    n = x.size
    area = np.full(n, 1.0 / n)
    w = 1.0 + 0.5 * np.sin(5 * x)
    act = np.ones(n, np.int32)
    if shape == "duplicates":
        act[:] = 0
        act[::300] = 1
        tgt = np.arange(n) % 300 == 0  # the copies sit on top of a source
    else:
        tgt = np.ones(n, bool)
    for kind, call in ((L.K_PLANE_BS, lambda p: ctx.plane_velocity(x, y, w, area, act, precision=p)),
                       (L.K_PLANE_GREEN, lambda p: ctx.plane_stream(x, y, w, area, act, precision=p))):
        got, pairs = _rows(call("fp32")), _all_pairs(ctx, kind, "fp32", lambda: call("fp32"))
        for g, r, e in zip(got, _rows(call("fp64")), pairs):
            # random points come closer than mesh points: as far off as the all-pairs sum is
            own = rel_err_max(e[tgt], r[tgt])
            assert rel_err_max(g[tgt], r[tgt]) < max(TOL32, 1.5 * own), (shape, own)


@pytest.mark.parametrize("bad", ["weight_inf", "weight_nan", "source_nan", "target_nan"])
def test_far_tiles_spread_non_finite_values_like_all_pairs(ctx, bad):
    x, y, z, zeta, area, act = (np.array(a, copy=True) for a in _sphere("mesh"))
    j = int(np.flatnonzero(act)[12345])
    if bad == "weight_inf":
        zeta[j] = np.inf
    elif bad == "weight_nan":
        zeta[j] = np.nan
    elif bad == "source_nan":
        x[j] = np.nan
    else:
        x[int(np.flatnonzero(act == 0)[777])] = np.nan

    def call():
        return ctx.bve_sphere_velocity(x, y, z, zeta, area, act, precision="fp32")

    # (the all-pairs kernel's error-free sums turn an infinite sum into NaN)
    for g, r in zip(_rows(call()), _all_pairs(ctx, L.K_SPHERE_BS, "fp32", call)):
        assert np.array_equal(np.isfinite(g), np.isfinite(r))
        if bad != "weight_inf":
            assert np.array_equal(np.isnan(g), np.isnan(r))


def test_far_tiles_split_leaves_no_trace(ctx):
    x, y, z, zeta, area, act = _sphere("mesh")
    ref = _rows(ctx.bve_sphere_velocity(x, y, z, zeta, area, act, precision="fp32"))
    try:
        for splits in (1, 3, 64):
            ctx.set_tuning(L.K_SPHERE_BS, "fp32", 0, 0, splits)
            for g, r in zip(_rows(ctx.bve_sphere_velocity(x, y, z, zeta, area, act, precision="fp32")), ref):
                assert rel_err_max(g, r) < 1e-13
    finally:
        ctx.set_tuning(L.K_SPHERE_BS, "fp32", 0, 0, 0)


def test_far_tiles_solver_and_graph(ctx):
    """One order per step, captured with it: replays equal eager steps."""
    x, y, z, zeta, area, act = _sphere("shuffled")
    kw = dict(rotation_rate=2 * np.pi, precision="fp32", project=True)
    a = BVESolver(ctx, x, y, z, zeta, area, act, **kw)
    b = BVESolver(ctx, x, y, z, zeta, area, act, use_graph=True, **kw)
    d = BVESolver(ctx, x, y, z, zeta, area, act, rotation_rate=2 * np.pi, precision="fp64", project=True)
    for k in range(3):
        for s in (a, b, d):
            s.timestep(0.005)
        sa, sb, sd = a.state(), b.state(), d.state()
        assert all(np.array_equal(sa[q], sb[q]) for q in sa), k
        if k == 0:
            assert rel_err_max((sa["u"], sa["v"], sa["w"]), (sd["u"], sd["v"], sd["w"])) < TOL32
    for s in (a, b, d):
        s.delete()


@pytest.mark.parametrize("graph", [False, True])
def test_far_tiles_batch(ctx, graph):
    """Problems on both sides of the rule in one batch, with a radius other than 1."""
    rng = np.random.default_rng(4)
    probs = []
    for level, radius in ((3, 1.0), (6, 2.5), (4, 1.0), (6, 1.0)):
        m = mesh.icosahedral_mesh(level, radius=radius)
        idx = rng.permutation(m.n)
        x, y, z = m.x[idx], m.y[idx], m.z[idx]
        probs.append(dict(x=x, y=y, z=z, relvort=ic.random_gaussian_vortices(rng, 2, x / radius, y / radius, z / radius),
                          area=m.area[idx], active=m.active[idx], radius=radius, rotation_rate=2 * np.pi))
    a = BVEBatch(ctx, probs, precision="fp32", project=True, use_graph=graph)
    b = BVEBatch(ctx, probs, precision="fp64", project=True)
    c = BVEBatch(ctx, probs, precision="fp32", project=True)
    c.set_tuning(4, 256, 16384)  # all pairs
    for s in (a, b, c):
        s.timestep(0.005)
    for ga, gb, gc in zip(*(s.split(s.state()) for s in (a, b, c))):
        ref = (gb["u"], gb["v"], gb["w"])
        assert rel_err_max((ga["u"], ga["v"], ga["w"]), ref) < TOL32
        assert rel_err_max((ga["u"], ga["v"], ga["w"]), (gc["u"], gc["v"], gc["w"])) < 2 * TOL32
        assert rel_err_max((ga["x"], ga["y"], ga["z"]), (gb["x"], gb["y"], gb["z"])) < TOL32
    for s in (a, b, c):
        s.delete()


# ------------------------------------------------------- culled PSE and SWE sums
def _ops(ctx, x, y, z, f, area, act, eps, prec, **kw):
    """PSE calls on the plane (z None) or the sphere: name -> (kind, call)."""
    if z is None:
        u, v = np.sin(2 * y) + x, np.cos(x) * y
        return {
            "pse8": (L.K_PSE8, lambda: ctx.pse_plane_laplacian(x, y, f, area, act, eps, order=8, precision=prec, **kw)),
            "pse2": (L.K_PSE2, lambda: ctx.pse_plane_laplacian(x, y, f, area, act, eps, order=2, precision=prec, **kw)),
            "gradient": (L.K_PSE_DERIV_PLANE, lambda: ctx.pse_plane_gradient(x, y, f, area, act, eps, precision=prec,
                                                                             **kw)),
            "second": (L.K_PSE_DERIV_PLANE, lambda: ctx.pse_plane_second_partials(x, y, u, v, area, act, eps,
                                                                                  precision=prec, **kw)),
            "interpolate": (L.K_PSE_INTERP_PLANE, lambda: ctx.pse_plane_interpolate(
                x, y, f, area, act, eps, 0.9 * x[::2] + 1e-3, 0.9 * y[::2], precision=prec)),
            "swe": (L.K_SWE_PLANE, lambda: ctx.swe_plane_rhs(x, y, f, 0.2 * f, 1.0 + 0.1 * x, 0.05 * y, area, act, eps,
                                                             precision=prec, **kw)),
        }
    return {
        "laplacian": (L.K_PSE_SPHERE8, lambda: ctx.pse_sphere_laplacian(x, y, z, f, area, act, eps, precision=prec,
                                                                        **kw)),
        "gradient": (L.K_PSE_DERIV_SPHERE, lambda: ctx.pse_sphere_gradient(x, y, z, f, area, act, eps, precision=prec,
                                                                           **kw)),
        "divergence": (L.K_PSE_DERIV_SPHERE, lambda: ctx.pse_sphere_divergence(x, y, z, y * z, x * x, z, area, act, eps,
                                                                               precision=prec, **kw)),
        "interpolate": (L.K_PSE_INTERP_SPHERE, lambda: ctx.pse_sphere_interpolate(x, y, z, f, area, act, eps, y[::3],
                                                                                  z[::3], x[::3], precision=prec)),
    }


# The terms are the all-pairs kernel's; only their order of summation differs: FP64
# to 1e-11 of the largest value, FP32 to 5e-5 (the bar of the forced shapes).
CULL_TOL = {"fp64": 1e-11, "fp32": 5e-5}


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("eps_h", [0.7, 2.0, 9.0])
def test_culled_plane_sums(ctx, prec, eps_h):
    """Kernel widths from under the spacing to the whole domain, a shuffled grid with
    passive particles and a block of targets."""
    x, y, area, h = mesh.grid_centres(131, 1.0, jitter=1e-3, seed=3)
    rng = np.random.default_rng(9)
    idx = rng.permutation(x.size)
    x, y, area = x[idx], y[idx], area[idx]
    f = np.exp(-4.0 * (x * x + y * y)) + 0.3 * x
    act = (rng.uniform(size=x.size) < 0.93).astype(np.int32)
    for kw in ({}, {"i0": 333, "i1": x.size - 70}):
        for name, (kind, call) in _ops(ctx, x, y, None, f, area, act, eps_h * h, prec, **kw).items():
            for g, r in zip(_rows(call()), _all_pairs(ctx, kind, prec, call)):
                assert rel_err_max(g, r) <= CULL_TOL[prec], (name, kw)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("eps", [0.01, 0.04])
def test_culled_sphere_sums(ctx, prec, eps):
    m = mesh.icosahedral_mesh(5)
    f = np.sin(3 * m.x) * m.y + m.z
    for name, (kind, call) in _ops(ctx, m.x, m.y, m.z, f, m.area, m.active, eps, prec).items():
        for g, r in zip(_rows(call()), _all_pairs(ctx, kind, prec, call)):
            assert rel_err_max(g, r) <= 4 * CULL_TOL[prec], name


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("where", ["source", "target"])
def test_culled_sums_spread_non_finite_values_like_all_pairs(ctx, prec, bad, where):
    x, y, area, h = mesh.grid_centres(120, 1.0, jitter=1e-3, seed=3)
    f = np.exp(-4.0 * (x * x + y * y))
    act = np.ones(x.size, np.int32)
    j = 7000
    if where == "target":
        act[j] = 0
    f[j] = bad
    for name, (kind, call) in _ops(ctx, x, y, None, f, area, act, 2 * h, prec).items():
        if name == "second":
            continue  # does not read f
        for g, r in zip(_rows(call()), _all_pairs(ctx, kind, prec, call)):
            assert np.array_equal(np.isfinite(g), np.isfinite(r)), name


# ------------------------------------------------------- shallow water on far tiles
def _swe(ctx, x, y, area, act, eps, **kw):
    vort, div = np.sin(3 * x) + y, np.cos(2 * y) * x

    def call(prec="fp32"):
        return ctx.swe_plane_rhs(x, y, vort, div, 1.0 + 0.1 * x, 0.05 * y, area, act, eps, precision=prec, **kw)

    return call


@pytest.mark.parametrize("shape", ["grid", "strip", "duplicates", "units"])
@pytest.mark.parametrize("eps_h", [2.0, 40.0])
def test_far_tiles_shallow_water(ctx, shape, eps_h):
    """Far tiles by the matrix products of f and f^2, the others by the culled sum
    (4e9 pairs on): shuffled, passive particles, a block of targets that starts inside
    a tile, and lengths at which f^2 would leave the normal numbers.  As far off the
    FP64 sums as the all-pairs kernel is, or within the FP32 bar."""
    rng = np.random.default_rng(11)
    x, y, area, h = mesh.grid_centres(270, 1.0, jitter=1e-3, seed=3)
    n = x.size
    if shape == "strip":
        x, y = rng.uniform(-50, 50, n), rng.uniform(-0.01, 0.01, n)
    elif shape == "duplicates":
        x, y = np.repeat(x[::300], 300), np.repeat(y[::300], 300)
        n = x.size
        area = area[:n]
    elif shape == "units":
        x, y, area, h = x * 1e-9, y * 1e-9, area * 1e-18, h * 1e-9
    idx = rng.permutation(n)
    x, y, area = x[idx], y[idx], area[idx]
    act = (rng.uniform(size=n) < 0.93).astype(np.int32)
    tgt = np.ones(n, bool)
    if shape == "duplicates":  # one active particle a point, compared on itself
        order = np.lexsort((y, x))
        act = np.zeros(n, np.int32)
        act[order[::300]] = 1
        tgt = act == 1
    kw = {"i0": 333, "i1": n - 70} if shape == "grid" else {}
    call = _swe(ctx, x, y, area, act, eps_h * h, **kw)
    got, again = _rows(call()), _rows(call())
    pairs = _all_pairs(ctx, L.K_SWE_PLANE, "fp32", call)
    for k, (g, e, r, a) in enumerate(zip(got, pairs, _rows(call("fp64")), again)):
        own = rel_err_max(e[tgt], r[tgt])
        assert rel_err_max(g[tgt], r[tgt]) < max(TOL32, 1.5 * own), (shape, k, own)
        assert np.array_equal(g, a, equal_nan=True)  # the passive copies sit on a source


@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("what", ["vort", "depth", "target"])
def test_far_shallow_water_spreads_non_finite_values_like_all_pairs(ctx, bad, what):
    x, y, area, h = mesh.grid_centres(256, 1.0, jitter=1e-3, seed=3)
    vort, depth = np.sin(3 * x) + y, 1.0 + 0.1 * x
    act = np.ones(x.size, np.int32)
    j = 7000
    if what == "target":
        act[j] = 0
    (vort if what == "vort" else depth)[j] = bad

    def call():
        return ctx.swe_plane_rhs(x, y, vort, 0.2 * vort, depth, 0.05 * y, area, act, 2 * h, precision="fp32")

    for g, r in zip(_rows(call()), _all_pairs(ctx, L.K_SWE_PLANE, "fp32", call)):
        assert np.array_equal(np.isfinite(g), np.isfinite(r))


# ------------------------------------------- tiles too small to change a sum
@pytest.mark.parametrize("field", ["patch", "jump", "lattice"])
@pytest.mark.parametrize("space", ["plane", "sphere"])
def test_tiles_passed_over_never_matter(ctx, field, space):
    """A tile is passed over only where adding it would round away, so every target keeps
    its own accuracy, however small its sum: a field that is zero but for a patch (sums
    down to 1e-290 around it), one that jumps by 1e200, and a regular lattice whose
    sums cancel.  FP64 against all pairs, each target by itself: 2^-53 of the sum of
    its terms' magnitudes times their number, for terms of one sign 1e-11 of the sum."""
    rng = np.random.default_rng(4)
    if space == "plane":
        x, y, area, h = mesh.grid_centres(128, 1.0, jitter=0.0 if field == "lattice" else 1e-3, seed=3)
        z, eps, r = None, 2 * h, np.hypot(x, y)
    else:
        m = mesh.icosahedral_mesh(5)
        x, y, z, area, eps, r = m.x, m.y, m.z, m.area, 0.03, np.arccos(np.clip(m.z, -1, 1))
    if field == "patch":
        f = np.where(r < 0.2, 1.0 + 0.1 * x, 0.0)
    elif field == "jump":
        f = np.where(x > 0.05, 1e100, 1e-100)
    else:
        f = np.ones(x.size)
    act = np.ones(x.size, np.int32) if z is None else m.active
    idx = rng.permutation(x.size)
    pts = (0.97 * x[idx], 0.97 * y[idx]) if z is None else (y[::3], z[::3], x[::3])
    if z is None:
        def interpolate():
            return ctx.pse_plane_interpolate(x, y, f, area, act, eps, *pts, precision="fp64")

        def lap():
            return ctx.pse_plane_laplacian(x, y, f, area, act, eps, order=2, precision="fp64")
        kinds = ((L.K_PSE_INTERP_PLANE, interpolate), (L.K_PSE2, lap))
    else:
        def interpolate():
            return ctx.pse_sphere_interpolate(x, y, z, f, area, act, eps, *pts, precision="fp64")
        kinds = ((L.K_PSE_INTERP_SPHERE, interpolate),)
    for kind, call in kinds:
        got, ref = np.asarray(call()), _all_pairs(ctx, kind, "fp64", call)[0]
        if field == "lattice" and kind == L.K_PSE2:  # zero terms: f_j - f_i
            assert not got.any() and not ref.any()
            continue
        seen = np.abs(ref) > 1e-290
        print(space, field, kind, "smallest", np.abs(ref[seen]).min(), "zeros", (~seen).sum())
        if kind == L.K_PSE2 and field == "jump":
            assert rel_err_max(got, ref) < 1e-11  # both signs within a target
        # the delta kernel changes sign where its cubic does, far inside the near tiles
        err = np.abs(got - ref)[seen] / np.abs(ref[seen])
        assert np.quantile(err, 0.99) < 1e-11 and err.max() < 1e-7
        assert np.abs(got[~seen]).max(initial=0.0) < 1e-289


@pytest.mark.parametrize("active", [0, 1, 1023, 1024, 1025, 2049, 20480])
def test_stream_source_totals(ctx, active):
    """The FP32 stream function adds the sources' total in FP64: none, one block of
    1,024 sources, a remainder, many.  FP64 sums of the same sources, the FP32 bar."""
    m = mesh.icosahedral_mesh(5)
    act = np.zeros(m.n, np.int32)
    act[np.flatnonzero(m.active)[:active]] = 1
    q = 1.0 + 0.5 * m.z  # one sign: the total is as large as it can be
    got = ctx.bve_sphere_stream(m.x, m.y, m.z, q, q + m.x, m.area, act, precision="fp32")
    ref = ctx.bve_sphere_stream(m.x, m.y, m.z, q, q + m.x, m.area, act, precision="fp64")
    for g, r in zip(got, ref):
        assert np.abs(g - r).max() <= 2e-6 * np.abs(r).max()


# ---------------------------------------- tiles on the line between near and far
def _clusters_on_the_far_line():
    """16 x 16 clusters of 256 points, each on a line along x inside its own cell of the
    order's curve, so that each is one tile: radius a (1 + 1e-6) about c, both multiples
    of 2^-24.  Half-widths and distances of every second pair of neighbours in a row,
    about 1/8 apart, are chosen so that the far rule, distance > 1.001 a_s + 2.002 a_t,
    holds by one way of rounding it with one fused multiply-add and not by the other."""
    f32 = np.float32
    rng = np.random.default_rng(8)

    def fma(a, b, c):
        return f32(float(a) * float(b) + float(c))  # the product is exact in 64 bits

    def radius(k):
        a = f32(k * 2.0**-24)
        return f32(np.sqrt(f32(a * a)) * f32(1.000001))

    def pair():
        while True:
            kt, d = int(rng.integers(690000, 710000)), 2**21 + int(rng.integers(-2000, 2000))
            ks = int(round(d / 1.001001)) - 2 * kt
            t, s, dist = radius(kt), radius(ks), f32(d * 2.0**-24)
            one = fma(s, f32(1.001), f32(f32(2.002) * t))
            two = fma(t, f32(2.002), f32(f32(1.001) * s))
            if (dist * dist > one * one) != (dist * dist > two * two):
                return kt, ks, d

    x, y = [], []
    for row in range(16):
        for col in range(0, 16, 2):
            kt, ks, d = pair()
            for side, k in enumerate((kt, ks)):
                u = np.rint(np.linspace(-1.0, 1.0, 256) * k) + side * d
                x.append(-1.0 + (col + 0.5) / 8 + u * 2.0**-24)
                y.append(np.full(256, -1.0 + row / 8))
    return np.concatenate(x), np.concatenate(y)


def test_tiles_on_the_far_line_belong_to_one_kernel(ctx):
    """Far and near tiles of the shallow-water sums are two kernels' work: every tile
    pair is summed once, also where its distance is the far rule's threshold to the last
    bit.  A cluster summed twice or not at all is off by 1e-3 and more."""
    x, y = _clusters_on_the_far_line()
    n = x.size
    idx = np.random.default_rng(1).permutation(n)
    x, y = x[idx], y[idx]
    area = np.full(n, 4.0 / n)
    call = _swe(ctx, x, y, area, np.ones(n, np.int32), 1e-3)
    for g, e, r in zip(_rows(call()), _all_pairs(ctx, L.K_SWE_PLANE, "fp32", call), _rows(call("fp64"))):
        own = rel_err_max(e, r)
        assert rel_err_max(g, r) < max(TOL32, 1.5 * own), own
    for kind, call in ((L.K_PLANE_BS, lambda p: ctx.plane_velocity(x, y, 1.0 + x, area, np.ones(n, np.int32),
                                                                   precision=p)),):
        for g, r in zip(_rows(call("fp32")), _rows(call("fp64"))):
            assert rel_err_max(g, r) < 4 * TOL32


# ------------------------------------------------------- lengths and weights of any unit
@pytest.mark.parametrize("length,weight", [(1e-13, 1.0), (1e-11, 1.0), (1e-6, 1e-15), (1e6, 1e-5), (1e18, 1.0),
                                           (3e19, 1.0)])
@pytest.mark.parametrize("space", ["plane", "sphere"])
def test_far_tiles_in_any_unit(ctx, space, length, weight):
    """Far tiles multiply weights by positions and squares by each other: lengths at which
    those products leave the normal numbers, where a pair of the all-pairs kernel does
    not.  As far off the FP64 sums as that kernel is, or within the FP32 bar."""
    if space == "plane":
        x, y, area, _ = mesh.grid_centres(270, 1.0, jitter=5e-4, seed=2)
        x, y, area, q, act = x * length, y * length, area * length**2, weight * (1 + 0.5 * np.sin(5 * x)), np.ones(
            x.size, np.int32)
        calls = ((L.K_PLANE_BS, lambda p: ctx.plane_velocity(x, y, q, area, act, precision=p)),
                 (L.K_PLANE_GREEN, lambda p: ctx.plane_stream(x, y, q, area, act, precision=p)))
    else:
        x, y, z, q, area, act = _sphere("mesh")
        x, y, z, q, area = x * length, y * length, z * length, q * weight, area * length**2
        i1 = 50000
        calls = ((L.K_SPHERE_BS, lambda p: ctx.bve_sphere_velocity(x, y, z, q, area, act, i1=i1, radius=length,
                                                                   precision=p)),
                 (L.K_SPHERE_GREEN, lambda p: ctx.bve_sphere_stream(x, y, z, q, q, area, act, i1=i1, radius=length,
                                                                    precision=p)))
    for kind, call in calls:
        got, pairs, exact = _rows(call("fp32")), _all_pairs(ctx, kind, "fp32", lambda: call("fp32")), _rows(call("fp64"))
        for g, e, r in zip(got, pairs, exact):
            assert np.array_equal(np.isfinite(g), np.isfinite(e))
            if np.isfinite(e).all():  # (logarithms of squares beyond the FP32 range are not)
                own = rel_err_max(e, r)
                assert rel_err_max(g, r) < max(TOL32, 1.5 * own), own


def test_far_shallow_water_with_weak_fields(ctx):
    """As above for the products c conj(Z)^2: lengths of 1e-5 and fields of 1e-14."""
    x, y, area, h = mesh.grid_centres(270, 1.0, jitter=1e-3, seed=3)
    s, act = 1e-5, np.ones(x.size, np.int32)
    vort, div = 1e-14 * (np.sin(3 * x) + y), 1e-14 * np.cos(2 * y) * x

    def call(prec="fp32"):
        return ctx.swe_plane_rhs(s * x, s * y, vort, div, 1.0 + 0.1 * x, 0.05 * y, s * s * area, act, 2 * s * h,
                                 precision=prec)

    for g, e, r in zip(_rows(call()), _all_pairs(ctx, L.K_SWE_PLANE, "fp32", call), _rows(call("fp64"))):
        own = rel_err_max(e, r)
        assert rel_err_max(g, r) < max(TOL32, 1.5 * own), own


# ------------------------------------------------------- groups of 64 source tiles
def _assert_culled(pairs):
    """Calls of fewer pairs take the all-pairs kernel (kCullMinPairs of lpm_pair.hip)."""
    assert pairs >= 1.5e8


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("eps_h", [2.0, 9.0])
@pytest.mark.parametrize("side,block", [(182, 5000), (520, 1000)])
def test_culled_plane_sums_over_groups(ctx, prec, eps_h, side, block):
    """From 512 source tiles on, groups of 64 are tested first: 518 tiles, the last group
    of 6, and 4,225, more than the 64 groups that one mask holds.  Shuffled, a block of
    targets, then one source that is not finite."""
    x, y, area, h = mesh.grid_centres(side, 1.0, jitter=0.2 / side, seed=3)
    n = x.size
    rng = np.random.default_rng(5)
    idx = rng.permutation(n)
    x, y, area = x[idx], y[idx], area[idx]
    f = np.exp(-4.0 * (x * x + y * y)) + 0.3 * x
    act = np.ones(n, np.int32)
    act[rng.permutation(n)[:50]] = 0
    _assert_culled((n - 50) * block)
    i0, eps = n // 3, eps_h * h
    px, py = rng.uniform(-1, 1, block), rng.uniform(-1, 1, block)
    calls = ((L.K_PSE8, lambda: ctx.pse_plane_laplacian(x, y, f, area, act, eps, order=8, i0=i0, i1=i0 + block,
                                                        precision=prec)),
             (L.K_PSE_DERIV_PLANE, lambda: ctx.pse_plane_gradient(x, y, f, area, act, eps, i0=i0, i1=i0 + block,
                                                                  precision=prec)),
             (L.K_PSE_INTERP_PLANE, lambda: ctx.pse_plane_interpolate(x, y, f, area, act, eps, px, py,
                                                                      precision=prec)))
    for kind, call in calls:
        for g, r in zip(_rows(call()), _all_pairs(ctx, kind, prec, call)):
            assert rel_err_max(g, r) <= CULL_TOL[prec], kind
    j = int(np.flatnonzero(act)[77])
    f[j] = np.inf
    for kind, call in calls:
        for g, r in zip(_rows(call()), _all_pairs(ctx, kind, prec, call)):
            assert np.array_equal(np.isfinite(g), np.isfinite(r)), kind


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("eps", [0.01, 0.04])
def test_culled_sphere_sums_over_groups(ctx, prec, eps):
    """5,120 source tiles (icosahedral level 7), a block of targets or points."""
    m = mesh.icosahedral_mesh(7)
    f = np.sin(3 * m.x) * m.y + m.z
    i0, i1 = 200001, 201000
    _assert_culled(int(m.active.sum()) * (i1 - i0))
    p = [np.ascontiguousarray(c[i0:i1]) for c in (m.y, m.z, m.x)]
    a = (m.area, m.active, eps)
    for kind, call in (
            (L.K_PSE_SPHERE8, lambda: ctx.pse_sphere_laplacian(m.x, m.y, m.z, f, *a, i0=i0, i1=i1, precision=prec)),
            (L.K_PSE_DERIV_SPHERE, lambda: ctx.pse_sphere_gradient(m.x, m.y, m.z, f, *a, i0=i0, i1=i1, precision=prec)),
            (L.K_PSE_INTERP_SPHERE, lambda: ctx.pse_sphere_interpolate(m.x, m.y, m.z, f, *a, *p, precision=prec))):
        for g, r in zip(_rows(call()), _all_pairs(ctx, kind, prec, call)):
            assert rel_err_max(g, r) <= 4 * CULL_TOL[prec], kind


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("eps_h", [0.7, 2.0, 4.0])
def test_culled_plane_interpolation(ctx, prec, eps_h):
    """Interpolation at as many points as there are sources, shuffled, with passive
    particles; then sources that are not finite."""
    x, y, area, h = mesh.grid_centres(131, 1.0, jitter=1e-3, seed=3)
    rng = np.random.default_rng(9)
    f = np.exp(-4.0 * (x * x + y * y)) + 0.3 * x
    act = (rng.uniform(size=x.size) < 0.93).astype(np.int32)
    idx = rng.permutation(x.size)
    px, py = 0.9 * x[idx] + 1e-3, 0.9 * y[idx]
    _assert_culled(int(act.sum()) * px.size)

    def call():
        return ctx.pse_plane_interpolate(x, y, f, area, act, eps_h * h, px, py, precision=prec)

    assert rel_err_max(call(), _all_pairs(ctx, L.K_PSE_INTERP_PLANE, prec, call)[0]) <= CULL_TOL[prec]
    act[7000] = 1
    for bad in (np.inf, np.nan):
        f[7000] = bad
        assert np.array_equal(np.isfinite(call()), np.isfinite(_all_pairs(ctx, L.K_PSE_INTERP_PLANE, prec, call)[0]))


# ------------------------------------------------------- wide kernels
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("order", ["grid", "shuffled", "two_far_clusters"])
def test_wide_plane_kernels_take_all_pairs(ctx, prec, order):
    """A kernel that reaches nearly all pairs has no tile to pass over: the sum is the
    all-pairs kernel's, bit for bit.  A narrow one is not."""
    x, y, area, h = mesh.grid_centres(140, 1.0, jitter=1e-3, seed=3)
    if order == "shuffled":
        idx = np.random.default_rng(1).permutation(x.size)
        x, y, area = x[idx], y[idx], area[idx]
    elif order == "two_far_clusters":
        x = np.where(x > 0, x + 1e5, x)
    f = np.exp(-4.0 * (x * x + y * y)) + y
    act = np.ones(x.size, np.int32)
    _assert_culled(x.size**2)
    r = {L.K_PSE8: 4, L.K_PSE_DERIV_PLANE: 2, L.K_PSE_INTERP_PLANE: 2} if prec == "fp64" else {
        L.K_PSE8: 2, L.K_PSE_DERIV_PLANE: 2, L.K_PSE_INTERP_PLANE: 2}

    def calls(eps):
        return ((L.K_PSE8, lambda: ctx.pse_plane_laplacian(x, y, f, area, act, eps, order=8, precision=prec)),
                (L.K_PSE_DERIV_PLANE, lambda: ctx.pse_plane_gradient(x, y, f, area, act, eps, precision=prec)),
                (L.K_PSE_INTERP_PLANE, lambda: ctx.pse_plane_interpolate(x, y, f, area, act, eps, 0.97 * x, 0.97 * y,
                                                                         precision=prec)))

    def forced(kind, call):
        ctx.set_tuning(kind, prec, r[kind], 256 if prec == "fp32" else 64, 0)
        try:
            return _rows(call())
        finally:
            ctx.set_tuning(kind, prec, 0, 0, 0)

    for kind, call in calls(0.8):
        same = all(np.array_equal(g, e) for g, e in zip(_rows(call()), forced(kind, call)))
        assert same == (order != "two_far_clusters"), kind  # half of the pairs are out of reach there
    for kind, call in calls(2 * h):
        assert not all(np.array_equal(g, e) for g, e in zip(_rows(call()), forced(kind, call))), kind
