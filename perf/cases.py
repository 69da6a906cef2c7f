"""
Performance cases: what users of harmonica_amd run, from single profiles to
the terrain models of regional surveys, through its public calls.

``listed()`` names the fixed cases, ``draw(rng)`` makes another one of the
same families.  ``prepare`` builds a case's inputs from a seed, ``run`` makes
one pass, ``work`` states the least bytes and operations of a pass and
``exact`` evaluates the same quantity without this package, in 64 bits or
better.

Families (host arrays in and out unless noted):

prism_host     prism_gravity, one field, default checks: scattered bodies of
               a 3D model, points in the caller's order
layer_host     the layer accessor's gravity: a terrain layer under a survey
prism_device   prism_fields_device: a terrain layer as explicit prisms, all
               arrays resident on the GPU
layer_device   layer_gravity_fields: several fields of a layer in one call
magnetic       prism_magnetic: a magnetised terrain
autograd       layer_gz with its backward pass: one step of an inversion
batched        BatchedPrismGz: many independent models of uneven sizes
points         point_fields_device: point masses, arrays on the GPU
tesseroid      tesseroid_gravity, default checks: a regional model
eqs_fit        EquivalentSources.fit on scattered data
eqs_predict    EquivalentSources.predict on a grid, from known coefficients
"""

import concurrent.futures
import math

import numpy as np
import torch

import harmonica_amd as hm
from harmonica_amd import workloads
from harmonica_amd._autograd import LayerGeometry, layer_gz
from harmonica_amd._batched import BatchedPrismGz
from harmonica_amd._forward import point_fields_device, prism_fields_device, to_device
from harmonica_amd._layer import layer_gravity_fields

FIELDS = ("potential", "g_e", "g_n", "g_z", "g_ee", "g_nn", "g_zz", "g_en", "g_ez", "g_nz")
G = 6.6743e-11
MEAN_RADIUS = 6371008.771415059


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # A profile over a handful of bodies: what an interactive forward
        # modelling session calls again and again.  Latency.
        {"name": "prism_gz_profile", "family": "prism_host", "field": "g_z", "prisms": 24,
         "points": 501},
        # A 3D model of odd size with a gradient field and its scan for
        # singular points, at scattered stations.
        {"name": "prism_gzz_bodies", "family": "prism_host", "field": "g_zz", "prisms": 20011,
         "points": 2999},
        # The terrain correction of a ground survey: 500 m cells, 64 x 64 points.
        {"name": "layer_gz_survey", "family": "layer_host", "field": "g_z", "n_east": 100,
         "n_north": 100, "spacing": 500.0, "aspect": 1.0, "obs_east": 64, "obs_north": 64,
         "height": 2100.0, "holes": 0.0},
        # The headline workload: 1,000,000 terrain prisms, 65,536 points.
        {"name": "prism_gz_terrain", "family": "prism_device", "field": "g_z", "n_east": 1000,
         "n_north": 1000, "spacing": 100.0, "aspect": 1.0, "obs_east": 256, "obs_north": 256,
         "height": 2500.0},
        # All ten fields of a layer for a gradiometry survey, cells not square.
        {"name": "layer_ten_fields", "family": "layer_device", "fields": "all", "n_east": 317,
         "n_north": 290, "spacing": 200.0, "aspect": 1.25, "obs_east": 120, "obs_north": 111,
         "height": 2500.0, "holes": 0.05},
        # The vector field of a magnetised terrain for an airborne survey.
        {"name": "magnetic_b_terrain", "family": "magnetic", "field": "b", "n_side": 300,
         "obs_east": 130, "obs_north": 101, "height": 2300.0},
        # One gradient step of a basement inversion (forward and backward).
        {"name": "layer_gz_gradient", "family": "autograd", "n_side": 200, "obs_side": 128},
        # Many independent models at once, as a stochastic inversion runs them.
        {"name": "batched_gz_models", "family": "batched", "models": 48, "sizes": 3,
         "prisms_lo": 1000, "prisms_hi": 200000, "points_lo": 1000, "points_hi": 50000},
        # Point masses of a discretised body on a survey grid.
        {"name": "point_gz_masses", "family": "points", "fields": "g_z", "masses": 300007,
         "points": 65536},
        # A regional tesseroid model under a satellite-height or airborne grid.
        {"name": "tesseroid_gz_region", "family": "tesseroid", "field": "g_z", "n_lon": 60,
         "n_lat": 50, "spacing": 0.5, "obs_lon": 67, "obs_lat": 61, "height": 10e3},
        # Equivalent sources fitted to a ground survey.
        {"name": "eqs_fit_survey", "family": "eqs_fit", "data": 6007, "damping": 10.0,
         "precision": "float64"},
        # Their prediction on the processing grid.
        {"name": "eqs_predict_grid", "family": "eqs_predict", "sources": 30011, "obs_east": 401,
         "obs_north": 367, "dtype": "float64"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _layer_sizes(rng, lo, hi, obs_lo, obs_hi, most):
    """Layer and grid sizes of at most ``most`` pairs, log-uniform."""
    while True:
        side, obs = _log_int(rng, lo, hi), _log_int(rng, obs_lo, obs_hi)
        case = {"n_east": side, "n_north": max(2, round(side * rng.uniform(0.7, 1.3))),
                "obs_east": obs, "obs_north": max(1, round(obs * rng.uniform(0.6, 1.4)))}
        if case["n_east"] * case["n_north"] * case["obs_east"] * case["obs_north"] <= most:
            return case


def draw(rng):
    family = rng.choice(["prism_host", "layer_host", "prism_device", "layer_device", "magnetic",
                         "autograd", "batched", "points", "tesseroid", "eqs_fit", "eqs_predict"])
    if family == "prism_host":
        return {"family": family, "field": rng.choice(["g_z", "g_z", "potential", "g_e", "g_zz",
                                                       "g_ez"]),
                "prisms": _log_int(rng, 8, 40000), "points": _log_int(rng, 50, 6000)}
    if family == "layer_host":
        case = _layer_sizes(rng, 20, 500, 8, 128, 2e9)
        return {"family": family, "field": rng.choice(["g_z", "g_z", "potential", "g_n", "g_nz"]),
                **case, "spacing": rng.uniform(100.0, 1000.0),
                "aspect": rng.choice([1.0, 1.0, 0.8, 1.5]), "height": rng.uniform(900.0, 3000.0),
                "holes": rng.choice([0.0, 0.1])}
    if family == "prism_device":
        case = _layer_sizes(rng, 64, 1000, 16, 256, 3e10)
        return {"family": family, "field": "g_z", **case, "spacing": rng.uniform(50.0, 400.0),
                "aspect": rng.choice([1.0, 1.0, 0.8, 1.5]), "height": rng.uniform(2100.0, 4000.0)}
    if family == "layer_device":
        case = _layer_sizes(rng, 50, 400, 16, 128, 2e9)
        return {"family": family, "fields": rng.choice(["all", "g_ee,g_nn,g_zz,g_en,g_ez,g_nz",
                                                        "g_e,g_n,g_z"]),
                **case, "spacing": rng.uniform(100.0, 1000.0),
                "aspect": rng.choice([1.0, 1.0, 0.8, 1.5]), "height": rng.uniform(2100.0, 4000.0),
                "holes": rng.choice([0.0, 0.05])}
    if family == "magnetic":
        return {"family": family, "field": rng.choice(["b", "b", "b_u", "b_e"]),
                "n_side": _log_int(rng, 30, 400), "obs_east": _log_int(rng, 10, 130),
                "obs_north": _log_int(rng, 10, 130), "height": rng.uniform(2100.0, 3000.0)}
    if family == "autograd":
        return {"family": family, "n_side": _log_int(rng, 24, 256),
                "obs_side": _log_int(rng, 16, 160)}
    if family == "batched":
        return {"family": family, "models": _log_int(rng, 4, 64), "sizes": rng.randrange(1000),
                "prisms_lo": 100,
                "prisms_hi": _log_int(rng, 1000, 100000), "points_lo": 100,
                "points_hi": _log_int(rng, 1000, 30000)}
    if family == "points":
        return {"family": family, "fields": rng.choice(["g_z", "g_z", "potential", "g_zz", "all"]),
                "masses": _log_int(rng, 300, 300000), "points": _log_int(rng, 100, 60000)}
    if family == "tesseroid":
        return {"family": family, "field": rng.choice(["g_z", "g_z", "potential"]),
                "n_lon": _log_int(rng, 6, 64), "n_lat": _log_int(rng, 6, 52),
                "spacing": rng.choice([0.25, 0.5, 1.0]), "obs_lon": _log_int(rng, 6, 70),
                "obs_lat": _log_int(rng, 6, 62), "height": rng.uniform(5e3, 250e3)}
    if family == "eqs_fit":
        return {"family": family, "data": _log_int(rng, 200, 7000),
                "damping": rng.choice([1.0, 10.0]),
                "precision": rng.choice(["float64", "float64", "mixed"])}
    return {"family": family, "sources": _log_int(rng, 200, 40000),
            "obs_east": _log_int(rng, 20, 400), "obs_north": _log_int(rng, 20, 400),
            "dtype": rng.choice(["float64", "float64", "float32"])}


# ------------------------------------------------------------------- inputs
def _rng(seed):
    return np.random.default_rng(seed)


def _surface(n_north, n_east, rng, lo, hi):
    """Fractal relief in [lo, hi]."""
    return workloads.fractal_surface(max(n_north, n_east, 2), rng, lo, hi)[:n_north, :n_east]


def _terrain(case, rng):
    """Centres, tops, densities and survey grid of a terrain layer."""
    dx = case["spacing"]
    dy = dx * case["aspect"]
    easting = dx / 2 + dx * np.arange(case["n_east"])
    northing = dy / 2 + dy * np.arange(case["n_north"])
    surface = _surface(case["n_north"], case["n_east"], rng, 0.0, 2000.0)
    density = rng.uniform(2600.0, 2800.0, surface.shape)
    if case.get("holes"):
        surface[rng.random(surface.shape) < case["holes"]] = np.nan
    ge = np.linspace(0.37 * dx, dx * (case["n_east"] - 0.41), case["obs_east"])
    gn = np.linspace(0.37 * dy, dy * (case["n_north"] - 0.41), case["obs_north"])
    E, N = np.meshgrid(ge, gn)
    return easting, northing, surface, density, (E, N, np.full(E.shape, case["height"]))


def _bodies(case, rng):
    """Scattered bodies of a 3D model and stations above them."""
    m, n = case["prisms"], case["points"]
    span = 20e3
    sides = rng.uniform(50.0, 600.0, (m, 3))
    centre = np.column_stack([rng.uniform(0, span, m), rng.uniform(0, span, m),
                              rng.uniform(-8e3, -400.0, m)])
    prisms = np.column_stack([centre[:, 0] - sides[:, 0] / 2, centre[:, 0] + sides[:, 0] / 2,
                              centre[:, 1] - sides[:, 1] / 2, centre[:, 1] + sides[:, 1] / 2,
                              centre[:, 2] - sides[:, 2] / 2, centre[:, 2] + sides[:, 2] / 2])
    coords = (rng.uniform(0, span, n), rng.uniform(0, span, n), rng.uniform(10.0, 800.0, n))
    return coords, prisms, rng.uniform(100.0, 500.0, m)


def _magnetised(case, rng):
    n = case["n_side"]
    easting = 50.0 + 100.0 * np.arange(n)
    surface = _surface(n, n, rng, 0.0, 2000.0)
    prisms = workloads.layer_to_prisms(easting, easting, surface, -5000.0)
    mag = workloads.terrain_magnetization(n, seed=int(rng.integers(1 << 30)))
    E, N = np.meshgrid(np.linspace(37.0, 100.0 * n - 41.0, case["obs_east"]),
                       np.linspace(37.0, 100.0 * n - 41.0, case["obs_north"]))
    return (E, N, np.full(E.shape, case["height"])), prisms, mag


def _tesseroids(case, rng):
    """A regional model and a grid whose lines miss the tesseroids' edges."""
    d, n_lon, n_lat = case["spacing"], case["n_lon"], case["n_lat"]
    west, south = -60.0 + rng.uniform(-5, 5), -30.0 + rng.uniform(-5, 5)
    W, S = np.meshgrid(west + d * np.arange(n_lon), south + d * np.arange(n_lat))
    top = _surface(n_lat, n_lon, rng, -3e3, 4e3)
    tess = np.column_stack([W.ravel(), (W + d).ravel(), S.ravel(), (S + d).ravel(),
                            np.full(W.size, MEAN_RADIUS - 30e3), (MEAN_RADIUS + top).ravel()])
    jitter = rng.uniform(0.01, 0.09, 2)
    lon = np.linspace(west, west + d * n_lon, case["obs_lon"]) + jitter[0]
    lat = np.linspace(south, south + d * n_lat, case["obs_lat"]) + jitter[1]
    E, N = np.meshgrid(lon, lat)
    return (E, N, np.full(E.shape, MEAN_RADIUS + case["height"])), tess, \
        rng.uniform(2470.0, 2870.0, W.size)


def _survey_data(case, rng):
    """Scattered gravity data of a few sources, with 1 mGal of noise."""
    n = case["data"]
    coords = (rng.uniform(0, 1e5, n), rng.uniform(0, 1e5, n), rng.uniform(500.0, 1500.0, n))
    data = rng.normal(0.0, 1.0, n)
    for _ in range(3):
        x, y, z = rng.uniform(0, 1e5), rng.uniform(0, 1e5), rng.uniform(3e3, 8e3)
        r2 = (coords[0] - x) ** 2 + (coords[1] - y) ** 2 + (coords[2] + z) ** 2
        data += rng.choice([-1.0, 1.0]) * 2e9 * (coords[2] + z) / r2**1.5
    return coords, data


def _sources(case, rng):
    m = case["sources"]
    points = (rng.uniform(0, 1e5, m), rng.uniform(0, 1e5, m), rng.uniform(-4000.0, -3000.0, m))
    E, N = np.meshgrid(np.linspace(0, 1e5, case["obs_east"]),
                       np.linspace(0, 1e5, case["obs_north"]))
    return (E, N, np.full(E.shape, 1000.0)), points, rng.normal(0.0, 1e3, m)


def _masses(case, rng):
    m, n = case["masses"], case["points"]
    points = (rng.uniform(0, 1e5, m), rng.uniform(0, 1e5, m), rng.uniform(-5e3, -100.0, m))
    side = max(1, int(math.isqrt(n)))
    coords = (rng.uniform(0, 1e5, n), np.sort(rng.uniform(0, 1e5, n)), np.full(n, 500.0)) \
        if side * side != n else tuple(
            a.ravel() for a in (*np.meshgrid(np.linspace(0, 1e5, side),
                                             np.linspace(0, 1e5, side)),
                                np.full((side, side), 500.0)))
    return coords, points, rng.uniform(1e8, 1e10, m)


def _models(case, seed):
    """Uneven models as workloads.batched_models makes them, their sizes fixed
    by the case and their contents by the seed."""
    sizes, rng = _rng(case["sizes"]), _rng(seed)
    models = []
    for _ in range(case["models"]):
        m, n = (int(round(np.exp(sizes.uniform(np.log(lo), np.log(hi))))) for lo, hi in
                ((case["prisms_lo"], case["prisms_hi"]), (case["points_lo"], case["points_hi"])))
        sides = rng.uniform(50.0, 2000.0, (m, 3))
        centre = np.column_stack([rng.uniform(-10e3, 10e3, (m, 2)), rng.uniform(-20e3, 0.0, m)])
        top = np.minimum(centre[:, 2] + sides[:, 2] / 2, 0.0)
        prisms = np.column_stack([centre[:, 0] - sides[:, 0] / 2, centre[:, 0] + sides[:, 0] / 2,
                                  centre[:, 1] - sides[:, 1] / 2, centre[:, 1] + sides[:, 1] / 2,
                                  top - sides[:, 2], top])
        coords = (rng.uniform(-10e3, 10e3, n), rng.uniform(-10e3, 10e3, n),
                  rng.uniform(100.0, 3000.0, n))
        models.append((coords, prisms, rng.normal(0.0, 300.0, m)))
    return models


def _field_list(case):
    return FIELDS if case["fields"] == "all" else tuple(case["fields"].split(","))


def prepare(case, seed):
    rng, family = _rng(seed), case["family"]
    if family == "prism_host":
        coords, prisms, density = _bodies(case, rng)
        return {"case": case, "args": (coords, prisms, density, case["field"])}
    if family in ("layer_host", "layer_device"):
        easting, northing, surface, density, coords = _terrain(case, rng)
        layer = hm.prism_layer((easting, northing), surface, -5000.0 if family == "layer_device"
                               else 0.0, properties={"density": density})
        return {"case": case, "layer": layer, "coords": coords}
    if family == "prism_device":
        easting, northing, surface, density, coords = _terrain(case, rng)
        prisms = workloads.layer_to_prisms(easting, northing, surface, -5000.0)
        return {"case": case, "coords": tuple(to_device(c.ravel()) for c in coords),
                "prisms": to_device(prisms), "density": to_device(density.ravel())}
    if family == "magnetic":
        coords, prisms, mag = _magnetised(case, rng)
        return {"case": case, "args": (coords, prisms, mag, case["field"])}
    if family == "autograd":
        w = workloads.inversion_layer(seed=seed, n_side=case["n_side"],
                                      n_obs_side=case["obs_side"])
        geometry = LayerGeometry(w["easting"], w["northing"], w["bottom"], w["coordinates"])
        return {"case": case, "geometry": geometry,
                "density": to_device(w["density"]).requires_grad_(),
                "top": to_device(w["top"]).requires_grad_(),
                "data": to_device(rng.normal(-100.0, 30.0, geometry.n_obs))}
    if family == "batched":
        return {"case": case, "batch": BatchedPrismGz(_models(case, seed))}
    if family == "points":
        coords, points, masses = _masses(case, rng)
        return {"case": case, "coords": [to_device(c) for c in coords],
                "points": [to_device(p) for p in points], "masses": to_device(masses)}
    if family == "tesseroid":
        coords, tess, density = _tesseroids(case, rng)
        return {"case": case, "args": (coords, tess, density, case["field"])}
    if family == "eqs_fit":
        coords, data = _survey_data(case, rng)
        return {"case": case, "coords": coords, "data": data}
    coords, points, coefs = _sources(case, rng)
    eqs = hm.EquivalentSources(points=points, dtype=case["dtype"])
    # a model fitted earlier and loaded again
    eqs.points_ = tuple(p.astype(case["dtype"]) for p in points)
    eqs.coefs_ = coefs
    return {"case": case, "eqs": eqs, "coords": coords}


# ------------------------------------------------------------------ one pass
def run(state):
    case = state["case"]
    family = case["family"]
    if family == "prism_host":
        coords, prisms, density, field = state["args"]
        return hm.prism_gravity(coords, prisms, density, field=field)
    if family == "layer_host":
        return state["layer"].prism_layer.gravity(state["coords"], field=case["field"])
    if family == "prism_device":
        return prism_fields_device(*state["coords"], state["prisms"], state["density"],
                                   (case["field"],))
    if family == "layer_device":
        return layer_gravity_fields(state["layer"], state["coords"], _field_list(case))
    if family == "magnetic":
        coords, prisms, mag, field = state["args"]
        return hm.prism_magnetic(coords, prisms, mag, field)
    if family == "autograd":
        gz = layer_gz(state["density"], state["top"], state["geometry"])
        misfit = 0.5 * ((gz - state["data"]) ** 2).sum()
        return (gz.detach(), *torch.autograd.grad(misfit, (state["density"], state["top"])))
    if family == "batched":
        return state["batch"].run()
    if family == "points":
        return point_fields_device(*state["coords"], *state["points"], state["masses"],
                                   _field_list(case))
    if family == "tesseroid":
        coords, tess, density, field = state["args"]
        return hm.tesseroid_gravity(coords, tess, density, field=field)
    if family == "eqs_fit":
        eqs = hm.EquivalentSources(damping=case["damping"], depth=4500.0,
                                   fit_precision=case["precision"])
        eqs.fit(state["coords"], state["data"])
        return eqs.coefs_, eqs.predict(state["coords"])
    return state["eqs"].predict(state["coords"])


# ---------------------------------------------------- the least work of a pass
#: Operations no sum over (source, point) pairs does without: the distance and
#: its inverse (three differences, their squares, a reciprocal square root to
#: 53 bits) and the accumulation.
PAIR = 20.0


def work(case):
    family = case["family"]
    if family in ("prism_host",):
        n, m = case["points"], case["prisms"]
        return {"bytes": 8.0 * (4 * n + 7 * m), "flops": 2 * PAIR * n * m}
    if family in ("layer_host", "layer_device", "prism_device"):
        n, m = case["obs_east"] * case["obs_north"], case["n_east"] * case["n_north"]
        fields = len(_field_list(case)) if family == "layer_device" else 1
        per = 7 if family == "prism_device" else 3
        return {"bytes": 8.0 * ((3 + fields) * n + per * m),
                "flops": (2 * PAIR + 8 * (fields - 1)) * n * m}
    if family == "magnetic":
        n, m = case["obs_east"] * case["obs_north"], case["n_side"] ** 2
        fields = 3 if case["field"] == "b" else 1
        return {"bytes": 8.0 * ((3 + fields) * n + 9 * m),
                "flops": (2 * PAIR + 8 * (fields - 1)) * n * m}
    if family == "autograd":
        n, m = case["obs_side"] ** 2, case["n_side"] ** 2
        return {"bytes": 8.0 * (5 * n + 5 * m), "flops": 2 * 2 * PAIR * n * m}
    if family == "batched":
        models = _models(case, 0)
        n = sum(c[0].size for c, _, _ in models)
        m = sum(d.size for _, _, d in models)
        return {"bytes": 8.0 * (4 * n + 7 * m),
                "flops": 2 * PAIR * sum(c[0].size * d.size for c, _, d in models)}
    if family == "points":
        n, m, fields = case["points"], case["masses"], len(_field_list(case))
        return {"bytes": 8.0 * ((3 + fields) * n + 4 * m),
                "flops": (PAIR + 5 * (fields - 1)) * n * m}
    if family == "tesseroid":
        n, m = case["obs_lon"] * case["obs_lat"], case["n_lon"] * case["n_lat"]
        return {"bytes": 8.0 * (4 * n + 7 * m), "flops": 8 * PAIR * n * m}
    if family == "eqs_fit":
        n = case["data"]
        return {"bytes": 8.0 * 6 * n, "flops": n**3 + n**3 / 3 + 2 * PAIR * n * n}
    n, m = case["obs_east"] * case["obs_north"], case["sources"]
    size = 4.0 if case["dtype"] == "float32" else 8.0
    return {"bytes": size * (4 * n + 4 * m), "flops": PAIR * n * m}


# ----------------------------------------- the same quantities, without the package
def _threads(fn, n, block):
    """fn(slice) over blocks of n points, on a few threads (numpy's loops
    release the interpreter lock), stacked along the last axis."""
    parts = [slice(i, min(n, i + block)) for i in range(0, n, block)]
    with concurrent.futures.ThreadPoolExecutor(16) as pool:
        return np.concatenate(list(pool.map(fn, parts)), axis=-1)


#: Signs and units of the fields (G in, harmonica's out).
_UNIT = {"potential": G, "g_e": 1e5 * G, "g_n": 1e5 * G, "g_z": -1e5 * G, "g_ee": 1e9 * G,
         "g_nn": 1e9 * G, "g_zz": 1e9 * G, "g_en": 1e9 * G, "g_ez": -1e9 * G, "g_nz": -1e9 * G}


def _prism_vertex_sums(x, y, z, fields):
    """Closed forms of one vertex (Nagy et al. 2000), in extended precision."""
    r = np.sqrt(x * x + y * y + z * z)
    need = set(fields)

    def log(a, b2):  # ln(a + r) without cancellation for a < 0
        return np.where(a >= 0, np.log(np.abs(a) + r), np.log(b2 / (r + np.abs(a))))

    lx = ly = lz = ax = ay = az = None
    if need & {"potential", "g_n", "g_z", "g_nz"}:
        lx = log(x, y * y + z * z)
    if need & {"potential", "g_e", "g_z", "g_ez"}:
        ly = log(y, x * x + z * z)
    if need & {"potential", "g_e", "g_n", "g_en"}:
        lz = log(z, x * x + y * y)
    if need & {"potential", "g_e", "g_ee"}:
        ax = np.arctan(y * z / (x * r))
    if need & {"potential", "g_n", "g_nn"}:
        ay = np.arctan(x * z / (y * r))
    if need & {"potential", "g_z", "g_zz"}:
        az = np.arctan(x * y / (z * r))
    out = {}
    if "potential" in need:
        out["potential"] = x * y * lz + y * z * lx + z * x * ly - (x * x * ax + y * y * ay
                                                                  + z * z * az) / 2
    if "g_e" in need:
        out["g_e"] = -(y * lz + z * ly - x * ax)
    if "g_n" in need:
        out["g_n"] = -(z * lx + x * lz - y * ay)
    if "g_z" in need:
        out["g_z"] = -(x * ly + y * lx - z * az)
    for name, value in (("g_ee", ax), ("g_nn", ay), ("g_zz", az)):
        if name in need:
            out[name] = -value
    for name, value in (("g_en", lz), ("g_ez", ly), ("g_nz", lx)):
        if name in need:
            out[name] = value
    return out


def _prism_sums(coords, prisms, weights, fields):
    """sum over prisms of weights[f] x vertex sums of field f, for every point:
    (len(fields), n).  ``weights``: one (m,) array per field."""
    ld = np.longdouble
    e, n, u = (np.ravel(c).astype(ld) for c in coords)
    W, E, S, N, B, T = (prisms[:, k].astype(ld) for k in range(6))
    weights = [np.asarray(w).astype(ld) for w in weights]

    def part(s):
        out = np.zeros((len(fields), s.stop - s.start), dtype=ld)
        for p0 in range(0, W.size, 256):
            q = slice(p0, p0 + 256)
            for i, xb in enumerate((E, W)):
                x = xb[q][None, :] - e[s, None]
                for j, yb in enumerate((N, S)):
                    y = yb[q][None, :] - n[s, None]
                    for k, zb in enumerate((T, B)):
                        z = zb[q][None, :] - u[s, None]
                        v = _prism_vertex_sums(x, y, z, fields)
                        sign = -1 if (i + j + k) % 2 else 1
                        for f, name in enumerate(fields):
                            out[f] += sign * (v[name] @ weights[f][q])
        return out

    with np.errstate(all="ignore"):
        return _threads(part, e.size, 32)


def _cost(fields):
    """Seconds per 1e9 (point, prism) pairs of _prism_sums on 16 threads."""
    return 8 * 9.0 * sum({"potential": 6, "g_e": 3, "g_n": 3, "g_z": 3}.get(f, 1) for f in fields)


def _prism_exact(coords, prisms, density, fields):
    pairs = np.size(coords[0]) * prisms.shape[0]
    if pairs / 1e9 * _cost(fields) > 15:
        return None
    sums = _prism_sums(coords, prisms, [density] * len(fields), fields)
    return np.stack([np.asarray(s * _UNIT[f], dtype=np.float64) for s, f in zip(sums, fields)])


def _inverse_distances(coords, points, coefs, fields=("potential",)):
    """Point-mass sums in 64 bits, G and units left out."""
    e, n, u = (np.ravel(c).astype(np.float64) for c in coords)
    p = [np.asarray(v, dtype=np.float64) for v in points]
    c = np.asarray(coefs, dtype=np.float64)

    def part(s):
        out = np.zeros((len(fields), s.stop - s.start))
        for p0 in range(0, c.size, 4096):
            q = slice(p0, p0 + 4096)
            d = [a[s, None] - b[q][None, :] for a, b in zip((e, n, u), p)]
            r2 = d[0] ** 2 + d[1] ** 2 + d[2] ** 2
            i1 = 1.0 / np.sqrt(r2)
            for f, name in enumerate(fields):
                if name == "potential":
                    k = i1
                elif name in ("g_e", "g_n", "g_z"):
                    k = -d["enz".index(name[-1])] * i1 / r2
                else:
                    a, b = ("enz".index(t) for t in name[2:])
                    k = (3 * d[a] * d[b] - (r2 if a == b else 0.0)) * i1 / (r2 * r2)
                out[f] += k @ c[q]
        return out

    return _threads(part, e.size, 64)


def _tesseroid_exact(coords, tess, density, field):
    """Adaptive discretisation and 2 x 2 x 2 Gauss-Legendre quadrature of the
    spherical kernels, with 1 - cos(psi) as haversines."""
    lon, lat, rad = (np.radians(np.ravel(c)) if k < 2 else np.ravel(c)
                     for k, c in enumerate(coords))
    ratio = 1.0 if field == "potential" else 2.5
    node = 1.0 / math.sqrt(3.0)

    def kernel(i, lo, la, r):
        hav = np.sin((lat[i] - la) / 2) ** 2 \
            + np.cos(lat[i]) * np.cos(la) * np.sin((lon[i] - lo) / 2) ** 2
        d = np.sqrt((rad[i] - r) ** 2 + 4 * rad[i] * r * hav)
        dz = rad[i] - r + 2 * r * hav
        return d, (1 / d if field == "potential" else dz / d**3)

    def part(s):
        out = np.zeros(s.stop - s.start)
        ii, jj = (a.ravel() for a in np.meshgrid(np.arange(s.start, s.stop),
                                                 np.arange(tess.shape[0]), indexing="ij"))
        w, e, so, no, bo, to = (tess[jj, k] for k in range(6))
        rho = density[jj]
        while ii.size:
            mid = [(a + b) / 2 for a, b in ((w, e), (so, no), (bo, to))]
            d, _ = kernel(ii, np.radians(mid[0]), np.radians(mid[1]), mid[2])
            l_lon = to * 2 * np.arcsin(np.cos(np.radians(mid[1])) * np.sin(np.radians(e - w) / 2))
            l_lat = to * np.radians(no - so)
            near = (d / l_lon < ratio) * 1 + (d / l_lat < ratio) * 2
            k = near == 0
            mass = rho * np.radians(e - w) * np.radians(no - so) * (to - bo) / 8
            for a in (-node, node):
                la = np.radians(mid[1] + a * (no - so) / 2)
                for b in (-node, node):
                    r = mid[2] + b * (to - bo) / 2
                    for c in (-node, node):
                        lo = np.radians(mid[0] + c * (e - w) / 2)
                        v = kernel(ii[k], lo[k], la[k], r[k])[1]
                        out += np.bincount(ii[k] - s.start, (mass * r**2 * np.cos(la))[k] * v,
                                           minlength=out.size)
            parts = []
            for code in (1, 2, 3):
                q = near == code
                lons = ((w, mid[0]), (mid[0], e)) if code & 1 else ((w, e),)
                lats = ((so, mid[1]), (mid[1], no)) if code & 2 else ((so, no),)
                for x0, x1 in lons:
                    for y0, y1 in lats:
                        parts.append([v[q] for v in (ii, x0, x1, y0, y1, bo, to, rho)])
            ii, w, e, so, no, bo, to, rho = (np.concatenate(v) for v in zip(*parts))
        return out

    return _threads(part, lon.size, 32)


def exact(case, seed):
    rng, family = _rng(seed), case["family"]
    if family == "prism_host":
        coords, prisms, density = _bodies(case, rng)
        out = _prism_exact(coords, prisms, density, (case["field"],))
        return None if out is None else out[0]
    if family in ("layer_host", "layer_device", "prism_device"):
        easting, northing, surface, density, coords = _terrain(case, rng)
        prisms = workloads.layer_to_prisms(easting, northing, surface,
                                           0.0 if family == "layer_host" else -5000.0)
        keep = ~np.isnan(surface.ravel())
        fields = _field_list(case) if family == "layer_device" else (case["field"],)
        out = _prism_exact(coords, prisms[keep], density.ravel()[keep], fields)
        if out is None:
            return None
        return out[0].reshape(coords[0].shape) if family == "layer_host" else out
    if family == "magnetic":
        coords, prisms, (me, mn, mu) = _magnetised(case, rng)
        # b_i = c_m sum_j M_j K_ij, K the second derivatives of the east-north-up frame
        terms = {"b_e": ((me, "g_ee"), (mn, "g_en"), (mu, "g_ez")),
                 "b_n": ((me, "g_en"), (mn, "g_nn"), (mu, "g_nz")),
                 "b_u": ((me, "g_ez"), (mn, "g_nz"), (mu, "g_zz"))}
        names = ("b_e", "b_n", "b_u") if case["field"] == "b" else (case["field"],)
        flat = [t for name in names for t in terms[name]]
        if coords[0].size * prisms.shape[0] / 1e9 * _cost([f for _, f in flat]) > 10:
            return None
        sums = [_prism_sums(coords, prisms, [w], (f,))[0] for w, f in flat]
        out = tuple(np.asarray(sum(sums[3 * k:3 * k + 3]) * 100, dtype=np.float64)
                    .reshape(coords[0].shape) for k in range(len(names)))  # 1e-7 x 1e9 nT
        return out if case["field"] == "b" else out[0]
    if family == "batched":
        models = _models(case, seed)
        if sum(c[0].size * d.size for c, _, d in models) / 1e9 * _cost(("g_z",)) > 15:
            return None
        outs = []
        for coords, prisms, density in models:
            order = _upload_order(coords)
            outs.append(_prism_exact(tuple(c[order] for c in coords), prisms, density,
                                     ("g_z",))[0])
        return np.concatenate(outs)
    if family == "points":
        coords, points, masses = _masses(case, rng)
        fields = _field_list(case)
        if coords[0].size * masses.size * len(fields) > 3e9:
            return None
        out = _inverse_distances(coords, points, masses, fields)
        return np.stack([o * _UNIT[f] for o, f in zip(out, fields)])
    if family == "tesseroid":
        coords, tess, density = _tesseroids(case, rng)
        if coords[0].size * tess.shape[0] > 1.5e7:
            return None
        out = _tesseroid_exact(coords, tess, density, case["field"])
        return (out * G * (1 if case["field"] == "potential" else 1e5)).reshape(coords[0].shape)
    if family == "eqs_fit":
        coords, data = _survey_data(case, rng)
        points = (coords[0], coords[1], coords[2] - 4500.0)
        jac = 1.0 / np.sqrt(sum((a[:, None] - b[None, :]) ** 2 for a, b in zip(coords, points)))
        scale = jac.std(axis=0)
        normal = (jac / scale).T @ (jac / scale)
        normal[np.diag_indices_from(normal)] += case["damping"]
        coefs = np.linalg.solve(normal, (jac / scale).T @ data) / scale
        return coefs, jac @ coefs
    if family == "eqs_predict":
        coords, points, coefs = _sources(case, rng)
        if coords[0].size * coefs.size > 5e9:
            return None
        dtype = case["dtype"]
        cast = [np.asarray(c).astype(dtype).astype(np.float64) for c in coords]
        pts = [p.astype(dtype) for p in points]
        out = _inverse_distances(cast, pts, coefs.astype(dtype))[0]
        return out.astype(dtype).reshape(coords[0].shape)
    return None  # autograd: its gradients have no counterpart outside the package


def _upload_order(coords):
    """The order in which BatchedPrismGz uploads (and returns) a model's
    points: boustrophedon strips of 64-point runs four times wider than tall."""
    e, n = coords[0], coords[1]
    h = np.sqrt(0.25 * 64 * np.ptp(e) * np.ptp(n) / e.size)
    strip = np.floor((n - n.min()) / h).astype(np.int64)
    return np.lexsort((np.where(strip % 2 == 0, e, -e), strip))
