"""
Far forms of the prism kernels (prism_far.h) against extended precision
(numpy.longdouble, 2^-63; the closed form for near pairs, quadrature for far
ones): models whose pairs fall on both
sides of every order's distance, tiles of 1 to 65 prisms (a tile holds 32),
equal and different rectangles, thin and zero-width rectangles, coordinates
far from the origin, more close pairs per wave than its list holds, left-out
layer cells and points with NaN.

Tolerances, before the first run: a far pair is off by a few roundings of
its two face terms w A / r (16 x 2^-53 of their sum; the truncation is below
4e-15 = 36 x 2^-53 of each), a closed pair by a few roundings of its terms
of size w r ln (64 x 2^-53 w r); the sums add the magnitudes (random signs
only make the error smaller).
"""

import numpy as np
import numpy.testing as npt
import pytest

pytestmark = pytest.mark.gpu

G = 6.6743e-11


@pytest.fixture(scope="module")
def hm():
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import harmonica_amd

    return harmonica_amd


def _gz_exact(coords, prisms, density):
    """(g_z, error bound) in mGal."""
    ld = np.longdouble
    e, n, u = (np.asarray(c, dtype=ld)[:, None] for c in coords)
    p = prisms.astype(ld)
    total = np.zeros((e.shape[0], p.shape[0]), dtype=ld)
    for i, x in enumerate((p[:, 1] - e, p[:, 0] - e)):
        for j, y in enumerate((p[:, 3] - n, p[:, 2] - n)):
            for k, z in enumerate((p[:, 5] - u, p[:, 4] - u)):
                r = np.sqrt(x * x + y * y + z * z)
                with np.errstate(all="ignore"):
                    lx = np.where(x >= 0, np.log(r + x), np.log((y * y + z * z) / (r - x)))
                    ly = np.where(y >= 0, np.log(r + y), np.log((x * x + z * z) / (r - y)))
                    v = -(x * ly + y * lx - z * np.arctan2(x * y, z * r))
                total += (-1) ** (i + j + k) * np.where(np.isfinite(v), v, 0)
    # arctan2 above is the principal arctangent only for z r > 0: undo its
    # branch for z < 0 (x y / (z r) is what the closed form takes)
    for i, x in enumerate((p[:, 1] - e, p[:, 0] - e)):
        for j, y in enumerate((p[:, 3] - n, p[:, 2] - n)):
            for k, z in enumerate((p[:, 5] - u, p[:, 4] - u)):
                branch = np.where(z < 0, np.where(x * y >= 0, 1, -1), 0)
                total -= (-1) ** (i + j + k) * z * branch * np.arctan2(ld(0), ld(-1))
    area = (p[:, 1] - p[:, 0]) * (p[:, 3] - p[:, 2])
    half2 = ((p[:, 1] - p[:, 0]) ** 2 + (p[:, 3] - p[:, 2]) ** 2) / 4
    dx, dy = (p[:, 0] + p[:, 1]) / 2 - e, (p[:, 2] + p[:, 3]) / 2 - n
    rt, rb = (np.sqrt(dx * dx + dy * dy + (z - u) ** 2) for z in (p[:, 5], p[:, 4]))
    far = np.minimum(rt, rb) ** 2 >= 12.0**2 * half2
    # far pairs, where the closed form cancels even in extended precision: the
    # integral over the faces by 10 x 10 Gauss-Legendre nodes ((1 / 12)^20)
    x10, w10 = np.polynomial.legendre.leggauss(10)
    quad = np.zeros_like(total)
    for xa, wa in zip(x10.astype(ld), w10.astype(ld)):
        for xb, wb in zip(x10.astype(ld), w10.astype(ld)):
            s = (dx + xa * (p[:, 1] - p[:, 0]) / 2) ** 2 + (dy + xb * (p[:, 3] - p[:, 2]) / 2) ** 2
            quad += wa * wb / 4 * (1 / np.sqrt(s + (p[:, 4] - u) ** 2)
                                   - 1 / np.sqrt(s + (p[:, 5] - u) ** 2))
    total = np.where(far, quad * area, total)  # upward component of the attraction
    w = np.abs(1e5 * G * density)
    area = np.abs(area)
    # the kernels take the far form from 12.9 half-diagonals
    far = np.minimum(rt, rb) ** 2 >= 12.9**2 * half2
    bound = np.where(far, 52 * (area / rt + area / rb), 64 * (np.maximum(rt, rb) + np.sqrt(half2)))
    eps = ld(2) ** -53
    return ((total * (-1e5 * G * density)).sum(axis=1).astype(float),
            (bound * w * eps).sum(axis=1).astype(float))


def _model(kind, m, rng):
    """(m, 6) prisms around the origin, sides about 100."""
    if kind == "grid":
        side = int(np.ceil(np.sqrt(m)))
        k = np.arange(m)
        x, y = 100.0 * (k % side), 100.0 * (k // side)
        sx = sy = np.full(m, 100.0)
    else:
        x, y = rng.uniform(0, 3e3, m), rng.uniform(0, 3e3, m)
        sx, sy = rng.uniform(20, 200, m), rng.uniform(20, 200, m)
        if kind == "thin":
            sx, sy[::3] = np.full(m, 1e-3), 300.0
    t = rng.uniform(-400, 0, m)
    return np.column_stack([x, x + sx, y, y + sy, t - rng.uniform(10, 3000, m), t])


@pytest.mark.parametrize("kind", ["grid", "different", "thin"])
@pytest.mark.parametrize("m", [1, 31, 32, 33, 65, 400])
def test_gz_all_distances(hm, kind, m):
    """Points at 30 m to 100 km from the model (all orders and the closed
    form), in two orders: along the distance, and shuffled so that every wave
    holds near and far points (its close pairs go through the list)."""
    rng = np.random.default_rng(m)
    prisms = _model(kind, m, rng)
    density = rng.uniform(100, 500, m)
    d, phi = np.geomspace(30.0, 1e5, 333), rng.uniform(0, 2 * np.pi, 333)
    coords = (50.0 + d * np.cos(phi), 50.0 + d * np.sin(phi), rng.uniform(5.0, 300.0, 333))
    expected, bound = _gz_exact(coords, prisms, density)
    got = hm.prism_gravity(coords, prisms, density, field="g_z")
    assert (np.abs(got - expected) <= bound).all()
    order = rng.permutation(333)
    mixed = hm.prism_gravity(tuple(c[order] for c in coords), prisms, density, field="g_z")
    assert (np.abs(mixed - expected[order]) <= bound[order]).all()
    npt.assert_allclose(mixed, got[order], rtol=0, atol=2.0 * bound.max())


def test_gz_far_from_the_origin(hm):
    """UTM-like coordinates: the far form's centre must not round to them."""
    rng = np.random.default_rng(3)
    prisms = _model("different", 300, rng)
    density = rng.uniform(100, 500, 300)
    coords = (rng.uniform(-2e4, 2e4, 200), rng.uniform(-2e4, 2e4, 200), rng.uniform(1, 900, 200))
    shift = np.array([612345.678, 612345.678, 7123456.789, 7123456.789, 0, 0])
    moved = prisms + shift  # rounds: take what the rounded bounds give
    coords = (coords[0] + shift[0], coords[1] + shift[2], coords[2])
    expected, bound = _gz_exact(coords, moved, density)
    got = hm.prism_gravity(coords, moved, density, field="g_z")
    assert (np.abs(got - expected) <= bound).all()


def test_gz_layer_skips_and_nan_points(hm):
    """A layer with NaN cells: the same as its remaining prisms; a NaN point
    gives NaN at its own place only."""
    rng = np.random.default_rng(4)
    e, n = np.arange(40) * 100.0, np.arange(37) * 80.0
    surface = rng.uniform(100, 900, (37, 40))
    surface[rng.random(surface.shape) < 0.3] = np.nan
    density = rng.uniform(2000, 3000, surface.shape)
    layer = hm.prism_layer((e, n), surface, 0.0, properties={"density": density})
    coords = [rng.uniform(-3e3, 7e3, 150), rng.uniform(-3e3, 7e3, 150), rng.uniform(950, 2e3, 150)]
    coords[1][7] = np.nan
    got = layer.prism_layer.gravity(coords, field="g_z")
    prisms = layer.prism_layer._to_prisms()
    keep = ~np.isnan(surface.ravel())
    expected, bound = _gz_exact(coords, prisms[keep], density.ravel()[keep])
    ok = np.arange(150) != 7
    assert np.isnan(got[7])
    assert (np.abs(got - expected) <= bound)[ok].all()


@pytest.mark.parametrize("shape,n_obs", [((2, 2), 1), ((9, 7), 63), ((5, 13), 65), ((33, 31), 129)])
def test_layer_gradient_is_the_adjoint(hm, shape, n_obs):
    """The VJP (far form, order 10 and closed form by distance; points from 40 m
    to 200 km) against the JVP, which takes the closed form for every pair:
    <J (a, b), v> = <(a, b), J^T v>, each term to the closed form's rounding
    (64 x 2^-53 of the pair's w r, as above, in sum over all pairs)."""
    import torch

    from harmonica_amd._autograd import LayerGeometry

    rng = np.random.default_rng(n_obs)
    e, n = 100.0 * np.arange(shape[1]), 130.0 * np.arange(shape[0])
    d, phi = np.geomspace(40.0, 2e5, n_obs), rng.uniform(0, 2 * np.pi, n_obs)
    coords = (d * np.cos(phi), d * np.sin(phi), rng.uniform(20.0, 500.0, n_obs))
    top = rng.uniform(-900, -10, shape)
    top.flat[0] = np.nan  # a left-out cell
    density = rng.uniform(200, 400, shape)
    geometry = LayerGeometry(e, n, np.full(shape, -2000.0), coords)
    dev = lambda a: torch.as_tensor(a).cuda()
    rho, T = dev(density), dev(top)
    a, b, v = rng.normal(size=shape), rng.normal(size=shape), rng.normal(size=n_obs)
    jv = geometry.jvp(rho, T, dev(a), dev(b)).cpu().numpy()
    ga, gb = (g.cpu().numpy() for g in geometry.vjp(rho, T, dev(v)))
    assert ga.flat[0] == 0.0 and gb.flat[0] == 0.0
    left, right = jv @ v, (a * ga).sum() + (b * gb).sum()
    E, N = np.meshgrid(e, n)
    r = np.sqrt((E.ravel()[:, None] - coords[0]) ** 2 + (N.ravel()[:, None] - coords[1]) ** 2
                + (2000.0 + coords[2]) ** 2)
    weight = 1e5 * G * (np.abs(a).ravel() + 400.0 * np.abs(b).ravel())
    assert abs(left - right) <= 64 * 2.0**-53 * (weight[:, None] * (r + 1.0) * np.abs(v)).sum()


TEN = ("potential", "g_e", "g_n", "g_z", "g_ee", "g_nn", "g_zz", "g_en", "g_ez", "g_nz")


def _fields_exact(coords, prisms, weights):
    """{field: (value, error bound)} of the ten fields (G, units and harmonica's
    signs left out) in extended precision, closed form vertex by vertex; the
    bound is 64 x 2^-53 of the terms' size r^2, r or 1 in sum over all pairs."""
    ld = np.longdouble
    e, n, u = (np.asarray(c, dtype=ld)[:, None] for c in coords)
    p = prisms.astype(ld)
    total = {f: 0 for f in TEN}
    for i, x in enumerate((p[:, 1] - e, p[:, 0] - e)):
        for j, y in enumerate((p[:, 3] - n, p[:, 2] - n)):
            for k, z in enumerate((p[:, 5] - u, p[:, 4] - u)):
                r = np.sqrt(x * x + y * y + z * z)
                lx, ly, lz = (np.where(a >= 0, np.log(r + np.abs(a)),
                                       np.log((b * b + c * c) / (r + np.abs(a))))
                              for a, b, c in ((x, y, z), (y, x, z), (z, x, y)))
                ax, ay, az = (np.arctan(b * c / (a * r)) for a, b, c in
                              ((x, y, z), (y, x, z), (z, x, y)))
                v = (x * y * lz + y * z * lx + z * x * ly
                     - (x * x * ax + y * y * ay + z * z * az) / 2,
                     -(y * lz + z * ly - x * ax), -(z * lx + x * lz - y * ay),
                     -(x * ly + y * lx - z * az), -ax, -ay, -az, lz, ly, lx)
                for f, value in zip(TEN, v):
                    total[f] = total[f] + (-1) ** (i + j + k) * value
    r = np.sqrt((np.abs((p[:, 0] + p[:, 1]) / 2 - e) + 300) ** 2
                + (np.abs((p[:, 2] + p[:, 3]) / 2 - n) + 300) ** 2
                + np.maximum(np.abs(p[:, 5] - u), np.abs(p[:, 4] - u)) ** 2)
    w = np.abs(weights)
    return {f: ((total[f] * weights).sum(axis=1).astype(float),
                (64 * r ** (2 if k == 0 else 1 if k < 4 else 0) * w).sum(axis=1).astype(float)
                * 2.0**-53) for k, f in enumerate(TEN)}


_UNIT = dict(zip(TEN, (1.0, 1e5, 1e5, -1e5, 1e9, 1e9, 1e9, 1e9, -1e9, -1e9)))


@pytest.mark.parametrize("kind", ["grid", "different"])
@pytest.mark.parametrize("m", [1, 31, 33, 70])
def test_all_fields_all_distances(hm, kind, m):
    """Single fields, the fused sets and the magnetic components at points above
    the model, below it, level with it and straight above one prism, from 40 m
    to 100 km: every order, the closed form, and waves that mix them."""
    from harmonica_amd._forward import prism_fields_device, to_device

    rng = np.random.default_rng(m)
    prisms = _model(kind, m, rng)
    rho = rng.uniform(100, 500, m)
    k = 200
    d, phi = np.geomspace(40.0, 1e5, k), rng.uniform(0, 2 * np.pi, k)
    up = np.r_[rng.uniform(5.0, 300.0, 80), rng.uniform(-4e3, -3.5e3, 60), rng.uniform(-300, -1, 60)]
    coords = [53.0 + d * np.cos(phi), 47.0 + d * np.sin(phi), up]
    up[::2] *= 5.0
    centre = prisms[0, [0, 2]] + 0.37 * (prisms[0, [1, 3]] - prisms[0, [0, 2]])
    coords = [np.r_[coords[0], np.full(20, centre[0])], np.r_[coords[1], np.full(20, centre[1])],
              np.r_[coords[2], np.geomspace(500.0, 3e4, 20)]]
    order = rng.permutation(k + 20)
    coords = [c[order] for c in coords]
    exact = _fields_exact(coords, prisms, G * rho)
    dev = [to_device(np.ascontiguousarray(c)) for c in coords]
    P, D = to_device(prisms), to_device(rho)
    for fields in (*((f,) for f in TEN), TEN[1:4], TEN[4:], TEN):
        got = prism_fields_device(*dev, P, D, fields).cpu().numpy()
        for f, row in zip(fields, got):
            value, bound = exact[f]
            assert (np.abs(row / _UNIT[f] - value) <= bound).all(), (f, len(fields))
    me, mn, mu = (rng.normal(size=m) for _ in range(3))
    terms = {"b_e": ("g_ee", "g_en", "g_ez"), "b_n": ("g_en", "g_nn", "g_nz"),
             "b_u": ("g_ez", "g_nz", "g_zz")}
    for name, fields in terms.items():
        parts = [_fields_exact(coords, prisms, w)[f] for w, f in zip((me, mn, mu), fields)]
        value, bound = (sum(p[q] for p in parts) for q in (0, 1))
        got = hm.prism_magnetic(coords, prisms, (me, mn, mu), name) / 100.0  # 1e-7 x 1e9
        assert (np.abs(got - value) <= bound).all(), name


@pytest.mark.parametrize("others", [0, 1, 40], ids=["alone", "tile_different", "two_tiles"])
@pytest.mark.parametrize("sides", [(100.0, 100.0), (100.0, 300.0), (1e-3, 300.0), (300.0, 1e-3)])
def test_gz_orders_near_their_limit(hm, sides, others):
    """One prism at 8.82 to 25 half-diagonals from its nearer face (the
    shortest distances of orders 12, 10 and 8), straight above, below and to
    the sides; `others` weightless prisms of other rectangles change what the
    tile stages.  Bound as above, 52 x 2^-53 of the two face terms."""
    ld = np.longdouble
    rng = np.random.default_rng(int(sides[0]) + others)
    a, b = sides
    top, bottom = -50.0, -250.0
    prism = np.array([[-a / 2, a / 2, -b / 2, b / 2, bottom, top]])
    half = np.hypot(a, b) / 2
    k = 300
    r = half * np.geomspace(8.82, 25.0, k)
    phi, mu = rng.uniform(0, 2 * np.pi, k), rng.uniform(0, 1, k)
    phi[::5], mu[1::7], mu[2::7] = np.arctan2(b, a), 1.0, 0.0
    s, z = r * np.sqrt(1 - mu * mu), r * mu
    # above the top half of the time, below the bottom the other
    up = np.where(np.arange(k) % 2 == 0, top + z, bottom - z)
    coords = (s * np.cos(phi), s * np.sin(phi), up)
    order = rng.permutation(k)
    coords = tuple(c[order] for c in coords)
    x10, w10 = np.polynomial.legendre.leggauss(10)  # error (1 / 8.8)^20
    exact = np.zeros(k, dtype=ld)
    e, n, u = (c.astype(ld) for c in coords)
    for xa, wa in zip(x10.astype(ld), w10.astype(ld)):
        for xb, wb in zip(x10.astype(ld), w10.astype(ld)):
            q = (xa * a / 2 - e) ** 2 + (xb * b / 2 - n) ** 2
            exact += wa * wb / 4 * (1 / np.sqrt(q + (bottom - u) ** 2)
                                    - 1 / np.sqrt(q + (top - u) ** 2))
    rt, rb = (np.sqrt(e * e + n * n + (f - u) ** 2) for f in (top, bottom))
    scale = 1e5 * G * 300.0 * a * b
    bound = 52 * ld(2) ** -53 * scale * (1 / rt + 1 / rb)
    more = _model("different", max(others, 1), rng)[:others]
    prisms, density = np.vstack([prism, more]), np.r_[300.0, np.zeros(others)]
    got = hm.prism_gravity(coords, prisms, density, field="g_z")
    assert (np.abs(got + scale * exact) <= bound).all()


@pytest.mark.parametrize("between", [0, 1, 23, 24, 25, 39, 40, 41, 63, 64])
def test_close_waves_with_general_lanes(hm, between):
    """A wave of 64 close points of which `between` lie between two planes of
    the prisms (those pairs are listed, the rest evaluated in place or listed
    by their number)."""
    rng = np.random.default_rng(between)
    prisms = np.array([[0.0, 100.0, 0.0, 80.0, -150.0, -50.0], [0.0, 100.0, 0.0, 80.0, -300.0, -160.0]])
    density = np.array([300.0, -200.0])
    e = np.r_[rng.uniform(5.0, 95.0, between), rng.uniform(110.0, 300.0, 64 - between)]
    coords = [e, rng.uniform(90.0, 200.0, 64), rng.uniform(10.0, 60.0, 64)]
    order = rng.permutation(64)
    coords = [c[order] for c in coords]
    exact = _fields_exact(coords, prisms, G * density)
    for field in TEN:
        got = hm.prism_gravity(tuple(coords), prisms, density, field=field) / _UNIT[field]
        value, bound = exact[field]
        assert (np.abs(got - value) <= bound).all(), field


def _device_fields(coords, prisms, density, fields):
    from harmonica_amd._forward import prism_fields_device, to_device

    dev = [to_device(np.ascontiguousarray(c)) for c in coords]
    return prism_fields_device(*dev, to_device(prisms), to_device(density), fields).cpu().numpy()


def test_bottom_above_top(hm):
    """Prisms given with bottom and top exchanged, as the calls without checks
    take them, are prisms of the opposite sign: for points above both planes
    and below both in every field, for points between them in the fields whose
    closed form needs no logarithm along z, beside the model (the branches of
    the logarithms and of the angles in front of a face are chosen for bottom
    <= top)."""
    from harmonica_amd._forward import to_device
    from harmonica_amd._magnetic import magnetic_fields_device

    rng = np.random.default_rng(8)
    prisms = _model("different", 40, rng)
    prisms[:, 4], prisms[:, 5] = -2000.0 - rng.uniform(0, 50, 40), -1000.0 + rng.uniform(0, 50, 40)
    density = rng.uniform(100, 500, 40)
    swapped = prisms[:, [0, 1, 2, 3, 5, 4]]
    n = 300
    d, phi = np.geomspace(50.0, 5e4, n), rng.uniform(0.05, 1.5, n)
    flat = (3300.0 + d * np.cos(phi), 3300.0 + d * np.sin(phi))
    for low, high, fields in ((-900.0, 500.0, TEN), (-4000.0, -2100.0, TEN),
                              (-1900.0, -1100.0, ("g_z", "g_ee", "g_nn", "g_zz", "g_ez", "g_nz"))):
        coords = [*flat, rng.uniform(low, high, n)]
        exact = _fields_exact(coords, prisms, -G * density)
        for chosen in ((f,) for f in fields):
            row = _device_fields(coords, swapped, density, chosen)[0]
            value, bound = exact[chosen[0]]
            assert (np.abs(row / _UNIT[chosen[0]] - value) <= bound).all(), (chosen, low)
        for chosen in (TEN[4:], TEN):
            rows = _device_fields(coords, swapped, density, chosen)
            for f, row in zip(chosen, rows):
                if f in fields:
                    value, bound = exact[f]
                    assert (np.abs(row / _UNIT[f] - value) <= bound).all(), (f, low)
        # magnetisations along e and u (b_e) and along n and u (b_n)
        dev = [to_device(np.ascontiguousarray(c)) for c in coords]
        me, mu, zero = density, density[::-1].copy(), np.zeros(40)
        for name, m, terms in (("b_e", (me, zero, mu), ("g_ee", "g_ez")),
                               ("b_n", (zero, me, mu), ("g_nn", "g_nz"))):
            parts = [_fields_exact(coords, prisms, -w)[f] for w, f in zip((me, mu), terms)]
            value, bound = (sum(p[q] for p in parts) for q in (0, 1))
            got = magnetic_fields_device(*dev, to_device(swapped), *(to_device(x) for x in m),
                                         (name,)).cpu().numpy()[0] / 100.0
            assert (np.abs(got - value) <= bound).all(), (name, low)


def test_prisms_without_area(hm):
    """A prism of zero width in both directions, which the device-level calls
    do not leave out, adds 0 at every point off its edges, to the rounding of
    the closed form's terms (64 x 2^-53 of w r^2, w r or w): straight above
    and below it, level with it and at its own height range.  So do its
    derivatives."""
    import ctypes

    import torch

    from harmonica_amd import _lib
    from harmonica_amd._forward import to_device
    from harmonica_amd._magnetic import magnetic_fields_device

    prisms = np.array([[10.0, 10.0, 20.0, 20.0, -300.0, -100.0]])
    e = np.r_[np.full(40, 10.0), np.full(20, 10.0), np.linspace(-50, 500, 40)]
    n = np.r_[np.full(40, 20.0), np.full(20, 25.0), np.linspace(-50, 500, 40)]
    u = np.r_[np.geomspace(0.5, 1e5, 20) - 100.0, -300.0 - np.geomspace(0.5, 1e5, 20),
              np.linspace(-400, 0, 20), np.linspace(-500, 500, 40)]
    coords = [e, n, u]
    ulp, r = 64 * 2.0**-53, np.hypot(np.hypot(e - 10, n - 20), np.abs(u + 200) + 100)
    for fields in (*((f,) for f in TEN), TEN[1:4], TEN[4:], TEN):
        for f, row in zip(fields, _device_fields(coords, prisms, np.array([300.0]), fields)):
            power = 2 if f == "potential" else 1 if f in TEN[1:4] else 0
            assert (np.abs(row / _UNIT[f]) <= ulp * G * 300.0 * r**power).all(), (f, fields)
    dev = [to_device(c) for c in coords]
    one = to_device(np.ones(1))
    for names in (("b_e",), ("b_n",), ("b_u",), ("b_e", "b_n", "b_u")):
        got = magnetic_fields_device(*dev, to_device(prisms), one, one, one, names)
        assert (np.abs(got.cpu().numpy()) <= 3 * 100.0 * ulp).all(), names
    v, grads = to_device(np.ones(e.size)), torch.full((2, 1), 7.0, dtype=torch.float64).cuda()
    nbytes = ctypes.c_size_t(0)
    _lib.check(_lib.lib().hmx_gz_grad_workspace_bytes(e.size, 1, ctypes.byref(nbytes)))
    ws = torch.empty(nbytes.value, dtype=torch.uint8, device="cuda")
    p = to_device(prisms)
    _lib.check(_lib.lib().hmx_prism_gz_vjp(*(_lib.ptr(c) for c in dev), _lib.ptr(v), e.size,
                                           _lib.ptr(p), 1, _lib.ptr(grads[0]), _lib.ptr(grads[1]),
                                           _lib.ptr(ws), nbytes.value, None))
    ga, gb = grads.cpu().numpy()[:, 0]
    assert abs(ga) <= ulp * r.sum() and abs(gb) <= ulp * e.size


@pytest.mark.parametrize("power", [45, -55])
def test_sizes_far_from_a_metre(hm, power):
    """A model scaled by 2^45 and by 2^-55: the potential scales by the
    square, accelerations by the first power, the tensor not at all.  The
    powers of the expansion would overflow there (the half-diagonal times the
    distance, and the inverse distance, to the twelfth)."""
    rng = np.random.default_rng(12)
    prisms = _model("different", 20, rng)
    density = rng.uniform(100, 500, 20)
    n = 130
    d, phi = np.geomspace(300.0, 2e4, n), rng.uniform(0, 2 * np.pi, n)
    coords = [1500.0 + d * np.cos(phi), 1500.0 + d * np.sin(phi), rng.uniform(5.0, 3e3, n)]
    exact = _fields_exact(coords, prisms, G * density)
    scale = 2.0**power
    scaled = [c * scale for c in coords]
    for fields in (*((f,) for f in TEN), TEN[1:4], TEN[4:], TEN):
        rows = _device_fields(scaled, prisms * scale, density, fields)
        for f, row in zip(fields, rows):
            value, bound = exact[f]
            size = scale ** (2 if f == "potential" else 1 if f in TEN[1:4] else 0)
            assert (np.abs(row / size / _UNIT[f] - value) <= bound).all(), (f, fields)


@pytest.mark.parametrize("where", [1e6, 1e9, 1e20, 1e300, np.inf, np.nan])
def test_one_point_far_away(hm, where):
    """The first of the points lies far from the others (a placeholder, say):
    theirs are as accurate as the closed form, 64 x 2^-53 of each pair's w r."""
    rng = np.random.default_rng(13)
    prisms = _model("different", 60, rng)
    density = rng.uniform(100, 500, 60)
    n = 200
    d, phi = np.geomspace(300.0, 2e4, n), rng.uniform(0, 2 * np.pi, n)
    # local coordinates with random mantissas: not multiples of the ulp of `where`
    coords = [1500.0 + d * np.cos(phi), 1500.0 + d * np.sin(phi), rng.uniform(5.0, 900.0, n)]
    exact = _fields_exact(coords, prisms, G * density)
    given = [np.r_[where, coords[0]], np.r_[where, coords[1]], np.r_[100.0, coords[2]]]
    for fields in (*((f,) for f in TEN), TEN[1:4], TEN[4:], TEN):
        rows = _device_fields(given, prisms, density, fields)
        for f, row in zip(fields, rows):
            value, bound = exact[f]
            assert (np.abs(row[1:] / _UNIT[f] - value) <= bound).all(), (f, fields)


@pytest.mark.parametrize("sides", [(100.0, 100.0), (100.0, 300.0)])
def test_gz_rectangles_nearly_equal(hm, sides):
    """Rectangles that share the constants of the chunk's first one though
    their sides differ by just under the tolerance, at 8.82 to 60
    half-diagonals: 52 x 2^-53 of the two face terms as above, and 2^-36 of
    the correction of order 2, at most (h/r)^2 / 3 of each."""
    ld = np.longdouble
    rng = np.random.default_rng(int(sides[1]))
    a, b = sides
    near = 1.0 + 2.0**-37.05  # of a side: just under 2^-36 of its square
    top, bottom = -50.0, -250.0
    first = np.array([-a / 2, a / 2, -b / 2, b / 2, bottom, top])
    a, b = a * near, b * near
    prism = np.array([-a / 2, a / 2, -b / 2, b / 2, bottom, top])
    a, b = prism[1] - prism[0], prism[3] - prism[2]
    half = np.hypot(a, b) / 2
    k = 400
    r = half * np.geomspace(8.82, 60.0, k)
    phi, mu = rng.uniform(0, 2 * np.pi, k), rng.uniform(0, 1, k)
    phi[::5], mu[1::7], mu[2::7] = np.arctan2(b, a), 1.0, 0.0
    s, z = r * np.sqrt(1 - mu * mu), r * mu
    up = np.where(np.arange(k) % 2 == 0, top + z, bottom - z)
    coords = (s * np.cos(phi), s * np.sin(phi), up)
    x10, w10 = np.polynomial.legendre.leggauss(10)
    exact = np.zeros(k, dtype=ld)
    e, n, u = (c.astype(ld) for c in coords)
    for xa, wa in zip(x10.astype(ld), w10.astype(ld)):
        for xb, wb in zip(x10.astype(ld), w10.astype(ld)):
            q = (xa * a / 2 - e) ** 2 + (xb * b / 2 - n) ** 2
            exact += wa * wb / 4 * (1 / np.sqrt(q + (bottom - u) ** 2)
                                    - 1 / np.sqrt(q + (top - u) ** 2))
    rt, rb = (np.sqrt(e * e + n * n + (f - u) ** 2) for f in (top, bottom))
    scale = 1e5 * G * 300.0 * a * b
    bound = scale * sum((52 * ld(2) ** -53 + ld(2) ** -36 * (half / x) ** 2 / 3) / x
                        for x in (rt, rb))
    got = _device_fields(coords, np.vstack([first, prism]), np.array([0.0, 300.0]), ("g_z",))[0]
    assert (np.abs(got + scale * exact) <= bound).all()


@pytest.mark.parametrize("kind", ["grid", "different"])
@pytest.mark.parametrize("m", [1, 33, 65])
def test_gz_order_12_in_tiles(hm, kind, m):
    """Points 250 m to 2 km from the model, where most pairs take the highest
    orders: pairs from 8.81 half-diagonals on to the far form's bound (52 x
    2^-53 of the two face terms), nearer ones to the closed form's."""
    rng = np.random.default_rng(100 + m)
    prisms = _model(kind, m, rng)
    density = rng.uniform(100, 500, m)
    d, phi = np.geomspace(250.0, 2e3, 256), rng.uniform(0, 2 * np.pi, 256)
    coords = (50.0 + d * np.cos(phi), 50.0 + d * np.sin(phi), rng.uniform(5.0, 1500.0, 256))
    expected, _ = _gz_exact(coords, prisms, density)
    e, n, u = (c[:, None] for c in coords)
    area = (prisms[:, 1] - prisms[:, 0]) * (prisms[:, 3] - prisms[:, 2])
    half = np.hypot(prisms[:, 1] - prisms[:, 0], prisms[:, 3] - prisms[:, 2]) / 2
    s = np.hypot((prisms[:, 0] + prisms[:, 1]) / 2 - e, (prisms[:, 2] + prisms[:, 3]) / 2 - n)
    rt, rb = (np.hypot(s, z - u) for z in (prisms[:, 5], prisms[:, 4]))
    far = np.minimum(rt, rb) >= 8.81 * half
    bound = np.where(far, 52 * area * (1 / rt + 1 / rb), 64 * (np.maximum(rt, rb) + half))
    bound = 2.0**-53 * (bound * 1e5 * G * density).sum(axis=1)
    for order in (np.arange(256), rng.permutation(256)):
        got = hm.prism_gravity(tuple(c[order] for c in coords), prisms, density, field="g_z")
        assert (np.abs(got - expected[order]) <= bound[order]).all()


def test_more_outputs_than_a_launch_has_threads(hm):
    """A reduction of 2^28 + 30 outputs (b_e, b_n, b_u of one prism at 2^28 / 3 +
    10 points): 16 waves per 64 outputs would pass the 2^32 threads of a
    launch.  The points repeat, and so do the values."""
    import torch

    from harmonica_amd._magnetic import magnetic_fields_device

    if torch.cuda.get_device_properties(0).total_memory < 32 << 30:
        pytest.skip("needs 10 GB")
    n, k = (1 << 28) // 3 + 11, 1009
    rng = np.random.default_rng(5)
    base = [torch.as_tensor(rng.uniform(lo, hi, k)).cuda() for lo, hi in
            ((-500, 500), (-500, 500), (10, 90))]
    coords = [b.repeat(n // k + 1)[:n].contiguous() for b in base]
    prism = torch.tensor([[-30.0, 40.0, -20.0, 60.0, -200.0, -50.0]], dtype=torch.float64).cuda()
    mag = [torch.tensor([v], dtype=torch.float64).cuda() for v in (1.0, -2.0, 0.5)]
    names = ("b_e", "b_n", "b_u")
    few = magnetic_fields_device(*base, prism, *mag, names)
    many = magnetic_fields_device(*coords, prism, *mag, names)
    # the far form's offsets have another origin in each workgroup: 2^-40 of
    # the largest value, 2^13 roundings
    assert torch.isfinite(few).all()
    tolerance = 2.0**-40 * few.abs().max()
    for start in (0, k, (n // k - 1) * k):
        assert (many[:, start:start + k] - few).abs().max() <= tolerance
    assert (many[:, (n // k) * k:] - few[:, :n % k]).abs().max() <= tolerance


@pytest.mark.parametrize("n,m", [(8192, 8), (8193, 16), (8193, 31), (8193, 32), (131072, 15),
                                 (131073, 3), (131073, 4)])
def test_few_prisms(hm, n, m):
    """Calls on both sides of the lines below which every pair takes the closed
    form (beyond 8192 points: 32 prisms, with the potential or g_z 16, and 4
    beyond 131,072 points; g_ee, g_nn and g_en alone at any number), explicit prisms, a layer and the magnetic field, to
    the closed form's bound."""
    import torch

    from harmonica_amd._forward import layer_fields_device, prism_fields_device, to_device
    from harmonica_amd._magnetic import magnetic_fields_device

    rng = np.random.default_rng(n + m)
    prisms = _model("different", m, rng)
    rho = rng.uniform(100, 500, m)
    coords = [rng.uniform(-3e3, 6e3, n), rng.uniform(-3e3, 6e3, n), rng.uniform(5.0, 900.0, n)]
    pick = np.unique(np.r_[0, n - 1, rng.integers(0, n, 250)])
    some = [c[pick] for c in coords]
    exact = _fields_exact(some, prisms, G * rho)
    dev, P, D = [to_device(c) for c in coords], to_device(prisms), to_device(rho)
    index = torch.as_tensor(pick).cuda()
    for fields in (*((f,) for f in TEN), TEN[1:4], TEN[4:], TEN, ("g_z", "g_zz")):
        got = prism_fields_device(*dev, P, D, fields)[:, index].cpu().numpy()
        for f, row in zip(fields, got):
            value, bound = exact[f]
            assert (np.abs(row / _UNIT[f] - value) <= bound).all(), (f, len(fields))
    mag = [rng.normal(size=m) for _ in range(3)]
    terms = {"b_e": ("g_ee", "g_en", "g_ez"), "b_n": ("g_en", "g_nn", "g_nz"),
             "b_u": ("g_ez", "g_nz", "g_zz")}
    got = magnetic_fields_device(*dev, P, *(to_device(x) for x in mag), tuple(terms))
    for row, (name, fields) in zip(got[:, index].cpu().numpy() / 100.0, terms.items()):
        parts = [_fields_exact(some, prisms, w)[f] for w, f in zip(mag, fields)]
        value, bound = (sum(p[q] for p in parts) for q in (0, 1))
        assert (np.abs(row - value) <= bound).all(), name
    # a layer of 2 x 3 cells, one of them left out
    e, nn = np.array([0.0, 200.0]), np.array([0.0, 150.0, 300.0])
    top = rng.uniform(-300, -10, (3, 2))
    density = rng.uniform(100, 500, (3, 2))
    density[1, 0] = np.nan
    cells = np.array([[x - 100, x + 100, y - 75, y + 75, -900.0, top[j, i]]
                      for i, x in enumerate(e) for j, y in enumerate(nn) if (j, i) != (1, 0)])
    weights = np.array([density[j, i] for i in range(2) for j in range(3) if (j, i) != (1, 0)])
    got = layer_fields_device(*dev, to_device(e), to_device(nn), to_device(np.full((3, 2), -900.0)),
                              to_device(top), to_device(density), TEN)[:, index].cpu().numpy()
    for f, row in zip(TEN, got):
        value, bound = _fields_exact(some, cells, G * weights)[f]
        assert (np.abs(row / _UNIT[f] - value) <= bound).all(), f


def test_few_prisms_at_their_edges(hm):
    """Singular points and points on faces in a call that takes the closed
    form: NaN exactly for the fields that are singular there, and the flags."""
    k = 2500  # 10,000 points
    import torch

    from harmonica_amd._forward import prism_fields_device, to_device

    prism = np.array([[0.0, 100.0, 0.0, 80.0, -150.0, -50.0]])
    # on an easting-parallel edge, a northing-parallel one, an upward one, a face
    coords = [np.tile(c, k) for c in ([50.0, 0.0, 100.0, 50.0], [0.0, 40.0, 80.0, 40.0],
                                      [-50.0, -50.0, -100.0, -50.0])]
    flags = torch.zeros(1, dtype=torch.int32).cuda()
    got = prism_fields_device(*(to_device(c) for c in coords), to_device(prism),
                              to_device(np.ones(1)), TEN, flags=flags).cpu().numpy()
    nan = np.isnan(got)
    expected = {"g_ee": (0, 1, 1, 0), "g_nn": (1, 0, 1, 0), "g_zz": (1, 1, 0, 0),
                "g_en": (0, 0, 1, 0), "g_ez": (0, 1, 0, 0), "g_nz": (1, 0, 0, 0)}
    for f, row in zip(TEN, nan):
        assert (row.reshape(k, 4) == np.array(expected.get(f, (0, 0, 0, 0)), bool)).all(), f
    assert int(flags.item()) == 0x3f0


@pytest.mark.parametrize("others", [0, 50])
def test_points_on_the_lines_of_edges(hm, others):
    """Points exactly on the lines of a prism's edges, from its corners to 10,000
    half-diagonals away: where an edge points away from them, ln(x + r) along
    it has the argument 0 and counts as 0, as in the oracle.  Alone, and as
    some points of waves that lie elsewhere; over one prism, and over others
    around it.  To 64 roundings of the oracle's terms, logarithms below 32 in
    magnitude and angles, in sum over all pairs."""
    import oracle

    rng = np.random.default_rng(others)
    prisms = np.vstack([[[0.0, 100.0, 0.0, 80.0, -150.0, -50.0]],
                        _model("different", max(others, 1), rng)[:others]])
    prisms[1:, 4:] -= 500.0
    density = rng.uniform(100, 500, len(prisms))
    d = np.geomspace(30.0, 6e5, 40)
    lines = []
    for low, high, axis in ((0, 100, 0), (0, 80, 1), (-150, -50, 2)):
        along = np.r_[high + d, low - d]
        corners = [c for a, c in enumerate(((0.0, 100.0), (0.0, 80.0), (-150.0, -50.0))) if a != axis]
        for first in corners[0]:
            for second in corners[1]:
                rest = [np.full(80, first), np.full(80, second)]
                rest.insert(axis, along)
                lines.append(np.array(rest))
    lines = np.concatenate(lines, axis=1)
    k = lines.shape[1]
    elsewhere = np.array([rng.uniform(-3e3, 3e3, k), rng.uniform(-3e3, 3e3, k),
                          rng.uniform(-50.0, 900.0, k)])
    mixed = np.concatenate([lines, elsewhere], axis=1)[:, rng.permutation(2 * k)]
    ulp = 64 * 2.0**-53 * 8 * 32
    for coords in (lines, mixed):
        expected = {f: oracle.prism_gravity(tuple(coords), prisms, density, f) for f in TEN[4:]}
        for chosen in (*((f,) for f in TEN[4:]), TEN[4:], TEN):
            rows = _device_fields(coords, prisms, density, chosen)
            for f, row in zip(chosen, rows):
                if f in expected:
                    error = np.abs(row - expected[f]).max()
                    assert error <= ulp * G * 1e9 * density.sum(), (f, len(chosen))
        mag = tuple(rng.normal(size=len(prisms)) for _ in range(3))
        for f in ("b_e", "b_n", "b_u"):
            error = np.abs(hm.prism_magnetic(tuple(coords), prisms, mag, f)
                           - oracle.prism_magnetic(tuple(coords), prisms, mag, f)).max()
            assert error <= ulp * 100.0 * np.abs(mag).sum(), f
