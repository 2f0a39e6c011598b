"""Rays with directions of their own take the source at the points around their
paths alone; the same rays repeated until the full table is the cheaper choice
take every point's (timing "render_listed" and "gradient_listed" say which).  The
two add the same FP32 products in another order (at most 64 terms here, 4e-6 of
the sum of their sizes; measured 2e-7).  Base and refined grids, open and
periodic, both ways to interpolate, rays that pass their lists."""
import numpy as np
import pytest

from at3d_amd import gradient as G
from at3d_amd import synthetic as S
from tests.scenes import interior_rays, rel_l2

pytestmark = pytest.mark.gpu

TIMES = 40


def _solved(bc, nx=41, ny=37, nz=25, **kw):
    w = S.cloud_field(nx=nx, ny=ny, nz=nz, dx=0.03, dz=0.9 / (nz - 1), z0=0.4, seed=3, nmu=8, nphi=16)
    w.bc = bc
    rte = S.make_rte(w, **kw)
    rte.solve(3, verbose=False)
    return w, rte


def _refined():
    w = S.cloud_field(nx=9, ny=8, nz=9, dx=0.05, dz=0.9 / 8, z0=0.4, seed=3, nmu=8, nphi=16)
    rte = S.make_rte(w, split_accuracy=0.03)
    rte.solve(40, verbose=False)
    assert rte.state_size("npts") > 4 * rte.plan_size("npts")
    return w, rte


def _tiled(rays):
    return {k: np.tile(v, TIMES) for k, v in rays.items()}


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("n", [255, 300, 321])
@pytest.mark.parametrize("single", [False, True])
def test_listed_points_match_full_table(n, single):
    w, rte = _solved("open")
    rays = interior_rays(w, n, seed=n)
    a = rte.integrate_to_sensor(dict(rays), single_scatter=single)["I"]
    assert rte.timing("render_listed") == 1.0
    b = rte.integrate_to_sensor(_tiled(rays), single_scatter=single)["I"].reshape(TIMES, n)
    assert rte.timing("render_listed") == 0.0
    assert np.all(b == b[0])
    assert rel_l2(a, b[0]) < 2e-6
    assert np.all(np.abs(a - b[0]) <= 1e-5 * np.abs(b[0]) + 1e-7)


@pytest.mark.filterwarnings("ignore")
def test_ray_past_its_list_takes_the_full_table():
    """A nearly horizontal ray around a thin periodic domain crosses more cells
    than its list holds."""
    n = 20
    w = S.lognormal_blob(n=n, dx=0.05, dz=0.04, radius=0.2, mean=0.02, nleg=64, bc="periodic", nmu=8, nphi=16)
    rte = S.make_rte(w)
    rte.solve(2, verbose=False)
    rays = interior_rays(w, 900, seed=2)
    rays["ray_mu"][:3] = [0.004, -0.004, 0.006]
    a = rte.integrate_to_sensor(dict(rays))["I"]
    assert rte.timing("render_listed") == 2.0
    b = rte.integrate_to_sensor(_tiled(rays))["I"].reshape(TIMES, 900)[0]
    assert rte.timing("render_listed") == 0.0
    assert rel_l2(a, b) < 2e-6


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("correct", [True, False])
def test_refined_grid_listed_points_match_full_table(correct):
    """Also where a cell starts with the values the ray left the last one with,
    which differ from its own on a face between cells of two sizes."""
    w, rte = _refined()
    rte._correctinterpolate = correct
    n = 1500
    rays = interior_rays(w, n, seed=5)
    a = rte.integrate_to_sensor(dict(rays))["I"]
    assert rte.timing("render_listed") == 1.0
    b = rte.integrate_to_sensor(_tiled(rays))["I"].reshape(TIMES, n)
    assert rte.timing("render_listed") == 0.0
    assert np.all(b == b[0])
    assert rel_l2(a, b[0]) < 2e-6


def _periodic():
    w = S.lognormal_blob(n=20, dx=0.05, dz=0.04, radius=0.2, mean=2.0, nleg=64, bc="periodic", nmu=8, nphi=16)
    rte = S.make_rte(w)
    rte.solve(5, verbose=False)
    return w, rte


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("make,n,low,flat,ess,route", [
    (lambda: _solved("open"), 300, 0.0, 0, True, 1), (lambda: _solved("open"), 300, 0.0, 0, False, 1),
    # (a list holds 62 cells here; from mu = 0.5 on a ray crosses at most 0.76 km x 1.73 / 0.05 km x 1.42 + 19 = 57)
    (_periodic, 900, 0.5, 0, True, 1), (_periodic, 900, 0.5, 3, True, 2), (_refined, 1500, 0.0, 0, True, 1)],
    ids=["open", "open_all", "periodic", "periodic_past_its_list", "refined"])
def test_gradient_from_listed_points_matches_full_table(make, n, low, flat, ess, route):
    w, rte = make()
    rays = interior_rays(w, n, seed=8)
    rays["ray_mu"] = np.maximum(np.abs(rays["ray_mu"]), low)
    rays["ray_mu"][:flat] = 0.01
    rays["measurement_data"] = np.random.default_rng(1).uniform(0.02, 0.2, n).astype(np.float32)
    names = list(rte.medium)
    unk = [(names[0], "extinction"), (names[0], "ssalb"), (names[-1], "extinction")]
    g, c, out = G.levis_approximation_grad(rte, rays, unk, exact_single_scatter=ess)
    assert rte.timing("gradient_listed") == route
    gt, ct, outt = G.levis_approximation_grad(rte, _tiled(rays), unk, exact_single_scatter=ess)
    assert rte.timing("gradient_listed") == 0.0
    assert rel_l2(out["I"], outt["I"][:n]) < 2e-6
    assert c == pytest.approx(ct / TIMES, rel=1e-5)
    for k in range(3):
        assert rel_l2(g[k], gt[k] / TIMES) < 1e-5
