"""The work a user of this framework has it do, as timed cases.

Four kinds of pass, all through ``at3d_amd.synthetic.make_rte`` (an ``RTE``),
``RTE.solve``, ``RTE.integrate_to_sensor``, the flux and spherical-harmonic
diagnostics and ``gradient.levis_approximation_grad``:

* ``solve``: a solver object that is kept solves its medium to
  ``solution_accuracy``, the fluxes, mean intensity, net fluxes and net flux
  divergence are read and the views rendered (I, and Q and U of a polarized
  solve with NSTOKES 3).
* ``cold``: a new medium, as every request of a serving loop and every step
  of a retrieval brings one: set-up, device state, solve, fluxes, release.
* ``render``: images of a solved medium.  Parallel-ray views share a
  direction per view; a perspective camera has a direction for every pixel.
* ``gradient``: cost, gradient (extinction and single-scattering albedo of
  every voxel) and forward pixels of a solved medium against measurements.

Media are the seeded fields of ``at3d_amd.synthetic``: a cloud (a -5/3
Gaussian field over Rayleigh scattering), the open lognormal blob of the
serving stream, the periodic lognormal blob, its polarized cloud, and a thin
random medium.  Angular resolutions are (NMU, NPHI) = (8, 16) .. (16, 32).
"""
import math

import numpy as np

from at3d_amd import gradient as G
from at3d_amd import sensor
from at3d_amd import synthetic as S

MAXITER = 100


def listed():
    return [
        # the periodic 16^3 lognormal blob at NMU 8: the smallest medium of
        # the framework's workloads and its periodic boundary condition
        dict(name="solve_periodic16", kind="solve", scene="periodic", nx=16, ny=16, nz=16, nmu=8,
             views=1, pixels=16),
        # the serving stream's smallest request at its coarsest angles:
        # iterations of tens of microseconds, where launches count
        dict(name="solve_blob32", kind="solve", scene="blob", nx=32, ny=32, nz=32, nmu=8,
             views=1, pixels=32),
        # the headline solve
        dict(name="solve_cloud64", kind="solve", scene="cloud", nx=64, ny=64, nz=40, nmu=16,
             views=1, pixels=64),
        # the serving stream's largest request
        dict(name="solve_blob96", kind="solve", scene="blob", nx=96, ny=96, nz=48, nmu=16,
             views=1, pixels=96),
        # the polarized workload: solve, then 9 views of 128 x 128 for I, Q, U
        dict(name="solve_polarized128", kind="solve", scene="polarized", nx=128, ny=128, nz=64, nmu=16,
             views=9, pixels=128),
        # a serving request whole, new medium to fluxes, at the middle angles
        dict(name="cold_blob48", kind="cold", scene="blob", nx=48, ny=48, nz=32, nmu=12, split=0.0),
        # adaptive cell splitting at the default accuracy, odd sizes
        dict(name="cold_adaptive17", kind="cold", scene="cloud", nx=17, ny=15, nz=12, nmu=8, split=0.03),
        # three parallel views of the small blob: a render bound by latency
        dict(name="render_periodic16", kind="render", scene="periodic", nx=16, ny=16, nz=16, nmu=8,
             views=3, pixels=32, camera=False),
        # the headline workload's nine views of 64 x 64
        dict(name="render_cloud64", kind="render", scene="cloud", nx=64, ny=64, nz=40, nmu=16,
             views=9, pixels=64, camera=False),
        # one camera of 61 x 61 pixels over the headline cloud: 3721 directions
        dict(name="render_camera64", kind="render", scene="cloud", nx=64, ny=64, nz=40, nmu=16,
             views=1, pixels=61, camera=True),
        # the differentiation workload: 3 views of 32 x 32 of the 16^3 blob
        dict(name="gradient_periodic16", kind="gradient", scene="periodic", nx=16, ny=16, nz=16, nmu=8,
             views=3, pixels=32, camera=False),
        # the largest row of the published gradient timings: 57024 points of a
        # thin random medium, overhead sun, 26 cameras of 13 x 13 pixels
        dict(name="gradient_cameras36", kind="gradient", scene="thin", nx=36, ny=36, nz=44, nmu=16,
             views=26, pixels=13, camera=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a kind, a medium and its sizes, log-uniform."""
    kind = rng.choice(["solve", "solve", "solve", "cold", "render", "render", "gradient", "gradient"])
    scenes = {"solve": ["periodic", "blob", "cloud", "cloud", "polarized"], "cold": ["blob", "cloud", "adaptive"],
              "render": ["periodic", "blob", "cloud", "polarized"],
              "gradient": ["periodic", "cloud", "thin", "thin"]}
    scene = rng.choice(scenes[kind])
    c = dict(kind=kind, scene=scene, nmu=rng.choice([8, 12, 16]))
    if scene == "periodic":
        n = rng.randint(9, 16)
        c.update(nx=n, ny=n, nz=n, nmu=8)
    elif scene == "adaptive":
        c.update(scene="cloud", split=0.03, nx=rng.randint(9, 18), ny=rng.randint(9, 16), nz=rng.randint(9, 12),
                 nmu=8)
    elif kind == "gradient":
        c.update(nx=_log(rng, 9, 36), ny=_log(rng, 9, 36), nz=_log(rng, 11, 44))
    else:
        c.update(nx=_log(rng, 12, 96), ny=_log(rng, 12, 96), nz=_log(rng, 10, 48))
    if kind == "cold":
        c.setdefault("split", 0.0)
    if kind != "cold":
        camera = kind != "solve" and scene != "polarized" and rng.random() < 0.5
        views = _log(rng, 1, 26 if camera and kind == "gradient" else 9)
        # a camera has as many directions as pixels
        most = 13 if camera and views > 4 else 29 if camera and views > 1 else 61 if camera else 96
        c.update(views=views, pixels=_log(rng, 7, most))
        if kind != "solve":
            c["camera"] = camera
    return c


def _medium(c, seed):
    """The case's seeded medium."""
    nx, ny, nz, nmu = c["nx"], c["ny"], c["nz"], c["nmu"]
    if c["scene"] == "periodic":
        return S.lognormal_blob(n=nx, radius=0.3 * nx / 16, nleg=64, seed=seed, nmu=nmu, nphi=2 * nmu)
    if c["scene"] == "blob":
        wl = float(np.random.default_rng(seed).uniform(0.55, 2.2))
        return S.serve_medium((nx, ny, nz), nmu, 2 * nmu, wl, seed)
    if c["scene"] == "cloud":
        # the headline cloud's layer (0.35 .. 1.325 km) on nz levels; coarse
        # grids keep the domain's width
        dx = 0.02 * max(1.0, 64.0 / max(nx, ny))
        return S.cloud_field(nx=nx, ny=ny, nz=nz, dx=dx, dz=0.975 / (nz - 1), z0=0.35, seed=seed, nmu=nmu,
                             nphi=2 * nmu)
    if c["scene"] == "polarized":
        return S.polarized_cloud_field(nx=nx, ny=ny, nz=nz, dz=1.26 / (nz - 1), seed=seed, nmu=nmu, nphi=2 * nmu)
    # the published gradient timings' medium: extinction uniform in 1e-6 .. 0.1
    # / km, random albedo, overhead sun
    rng = np.random.default_rng(seed)
    ext = rng.uniform(1e-6, 0.1, (nx, ny, nz)).astype(np.float32)
    alb = rng.uniform(0.5, 1.0, (nx, ny, nz)).astype(np.float32)
    z = np.linspace(0.0, 1.1, nz).astype(np.float32)
    return S.Workload("thin", 0.9 / nx, 0.9 / nx, z, [(ext, alb, S.hg_legendre(0.85, 64))], nmu=nmu, nphi=2 * nmu,
                      solarmu=-1.0)


def _rte(c, w):
    if c["scene"] == "polarized":
        return S.make_rte(w, max_total_mb=60000.0, adapt_grid_factor=1.0)
    return S.make_rte(w, split_accuracy=c.get("split", 0.0))


def _sensor(c, w):
    """Parallel views across the azimuth plane, or cameras on a dome."""
    n, px = c["views"], c["pixels"]
    if not c.get("camera", False):
        zen = np.linspace(-60.0, 60.0, n) if n > 1 else [0.0]
        return S.view_rays(w, [(abs(t), 0.0 if t >= 0 else 180.0) for t in zen], px, px)
    x0, y0, z0, x1, y1, z1 = S.domain_box(w)
    look = np.array([(x0 + x1) / 2, (y0 + y1) / 2, (z0 + z1) / 2])
    size = max(x1 - x0, y1 - y0, z1 - z0)
    out = []
    for k in range(n):
        zen = np.deg2rad(55.0) * np.sqrt((k + 0.5) / n)
        az = 2.399963 * k
        pos = look + 1.8 * size * np.array([np.sin(zen) * np.cos(az), np.sin(zen) * np.sin(az), np.cos(zen)])
        out.append(sensor.perspective_projection(w.wavelength, 30.0, px, px, pos, look, [0.0, 1.0, 0.01]))
    return {k: np.concatenate([s[k] for s in out]) for k in ("ray_x", "ray_y", "ray_z", "ray_mu", "ray_phi")}


def prepare(case, seed):
    w = _medium(case, seed)
    s = dict(case=case, w=w)
    if case["kind"] == "cold":
        return s
    s["rte"] = _rte(case, w)
    s["rays"] = _sensor(case, w)
    if case["kind"] != "solve":
        s["rte"].solve(MAXITER, verbose=False)
    if case["kind"] == "gradient":
        # measured radiances: a smooth level with pixel-to-pixel variation
        rng = np.random.default_rng(seed + 1)
        n = s["rays"]["ray_x"].size
        s["rays"]["measurement_data"] = (0.08 * np.exp(0.4 * rng.standard_normal(n))).astype(np.float32)
        sp = list(s["rte"].medium)[0]
        s["unknowns"] = [(sp, "extinction"), (sp, "ssalb")]
    return s


def _fields(rte):
    f, h = rte.fluxes, rte.spherical_harmonics
    out = {k: f[k] for k in ("flux_down", "flux_up", "flux_direct")}
    out["mean_intensity"] = h["mean_intensity"]
    # the net flux as one vector field (Fy is nearly zero: the sun lies in x-z)
    out["net_flux"] = np.stack([h["Fx"], h["Fy"], h["Fz"]])
    out["net_flux_div"] = rte.net_flux_divergence["net_flux_div"]
    return out


def run(state):
    kind = state["case"]["kind"]
    if kind == "cold":
        rte = _rte(state["case"], state["w"])
        rte.solve(MAXITER, verbose=False)
        # on an adaptive grid the fields are read on the base grid
        out = {k: v for k, v in rte.fluxes.items() if k.startswith("flux")}
        rte.release()
        return out
    rte = state["rte"]
    if kind == "solve":
        rte.solve(MAXITER, verbose=False)
        out = _fields(rte)
        img = rte.integrate_to_sensor(dict(state["rays"]))
        out.update({k: img[k] for k in ("I", "Q", "U") if k in img})
        return out
    if kind == "render":
        img = rte.integrate_to_sensor(dict(state["rays"]))
        return {k: img[k] for k in ("I", "Q", "U") if k in img}
    grad, cost, img = G.levis_approximation_grad(rte, state["rays"], state["unknowns"])
    return {"gradient": grad, "cost": cost, "I": img["I"]}


def work(case):
    """Per iteration, the spherical-harmonic fields (source, radiance, previous
    source change) and the discrete-ordinate fields (source, radiance) are each
    written by one step and read whole by the next; transforms in their
    separable form (a Legendre sum per azimuthal order, then an FFT), about 30
    operations per point and ordinate for the sweep and 20 per harmonic for the
    source.  A ray needs the extinction and source of the points around the
    cells it crosses, a ray direction of its own the harmonic sum at each."""
    nmu = case["nmu"]
    nlm, nang = nmu * nmu, 1.4 * nmu * nmu
    nst = 3 if case["scene"] == "polarized" else 1
    npts = case["nx"] * case["ny"] * case["nz"]
    iters = {"periodic": 16, "blob": 11, "cloud": 8, "polarized": 10, "thin": 4}[case["scene"]]
    io = 4.0 * npts * (2 * 2 + 8)
    b, f = 0.0, 0.0
    if case["kind"] in ("solve", "cold"):
        if case.get("split", 0.0) > 0:
            npts, iters = 3 * npts, 14
        b += io + 4.0 * npts * nst * iters * (6 * nlm + 4 * nang)
        f += npts * nst * iters * (4.0 * nlm * nmu + 10.0 * nang * math.log2(2 * nmu) + 30 * nang + 20 * nlm)
    if "views" in case:
        rays = float(case["views"] * case["pixels"] ** 2)
        cells = rays * 1.5 * (case["nx"] + case["ny"] + case["nz"]) / 2
        camera = case.get("camera", False)
        grad = 6 if case["kind"] == "gradient" else 1
        seen = min(npts * (case["views"] if not camera else rays), cells * 4.0)   # (point, direction) pairs
        b += 4.0 * npts * nst * nlm + rays * (28 + 4 * nst) + grad * 16.0 * npts
        f += nst * seen * (2.0 * nlm + 4 * nmu) * (2 if grad > 1 else 1) + grad * nst * cells * 150
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Four times the largest difference seen between the level-ordered (FP32
    steps) and the point-ordered (FP64 steps) sweep over the listed cases and
    14 drawn ones: 1.4e-6 of a field of a solve, 4e-6 of the nearly vanishing U
    of a polarized one in the principal plane.  With adaptive splitting a cell
    whose criterion lies at the threshold to rounding divides in one and not
    in the other, which changes the fields around it."""
    if case.get("split", 0.0) > 0:
        return {"rel": 3e-4, "max": 2e-2}
    if case["scene"] == "polarized":
        return {"rel": 2e-5, "max": 5e-4}
    return {"rel": 6e-6, "max": 2e-4}


def exact(case, seed):
    """None: what these calls return is the converged solution of the
    discretised radiative-transfer iteration (and images of it), which has no
    closed form; a plain 64-bit solver of it takes far over 20 seconds."""
    return None
