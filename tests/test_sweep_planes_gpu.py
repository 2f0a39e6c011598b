"""The plane-ordered sweep of open grids against the point-ordered sweep (FP64
steps): FP32 cell integrals, so DO radiances, DO sources and SH sources agree to
2e-6 after three iterations, as the level-ordered ring's do.  Grids whose
ordinates go by z, by x and by y, odd sizes, uneven layers, planes of one point
row up to several points per thread, planes just past a thread count."""
import numpy as np
import pytest

from at3d_amd import synthetic as S
from tests.scenes import pol_blob, rel_l2

pytestmark = [pytest.mark.gpu, pytest.mark.filterwarnings("ignore:solution did not converge")]


def _cloud(nx, ny, nz, dx=0.05, dz=0.05, nmu=8, seed=3, dy=None, z=None, sky=0.0):
    w = S.cloud_field(nx=nx, ny=ny, nz=nz, dx=dx, dz=dz, z0=0.5 - 0.1 * dz * nz, seed=seed, nmu=nmu, nphi=2 * nmu)
    if dy is not None:
        w.dely = dy
    if z is not None:
        w.z = np.asarray(z, np.float32)
    return w


def _uneven(n):
    # layers from 0.8 to 1.2 times the mean
    d = 0.01 * (1.0 + 0.2 * np.sin(np.arange(n - 1)))
    return 0.6 + np.concatenate([[0.0], np.cumsum(d)])


GRIDS = {
    "2x2x2": lambda: _cloud(2, 2, 2), "3x2x5": lambda: _cloud(3, 2, 5), "2x3x17": lambda: _cloud(2, 3, 17),
    "flat_layers_by_z": lambda: _cloud(9, 11, 13, dx=0.3, dz=0.03),
    "tall_layers_by_sides": lambda: _cloud(13, 9, 7, dx=0.02, dz=0.15),
    "by_y": lambda: _cloud(8, 15, 9, dx=0.06, dy=0.02, dz=0.05), "by_x": lambda: _cloud(15, 8, 9, dx=0.02, dy=0.06),
    "uneven_layers_by_z": lambda: _cloud(7, 9, 12, dx=0.5, z=_uneven(12)),
    "l15": lambda: _cloud(17, 15, 12, nmu=16), "shared_edges": lambda: _cloud(12, 12, 12, dx=0.05, dz=0.05, nmu=16),
    "33x31x20": lambda: _cloud(33, 31, 20, dx=0.02, dz=0.03), "45x46x25": lambda: _cloud(45, 46, 25, dx=0.02, dz=0.03),
    "52x53x40": lambda: _cloud(52, 53, 40, dx=0.03, dz=0.02), "55x50x60": lambda: _cloud(55, 50, 60, dx=0.03, dz=0.03),
    "64x64x9": lambda: _cloud(64, 64, 9, dx=0.02, dz=0.1),
    # planes of several strips: of unequal rows, across z, x and y, all three, of two points to four a thread
    "strips_66x63x9": lambda: _cloud(66, 63, 9, dx=0.02, dz=0.1),
    "strips_97x96x6": lambda: _cloud(97, 96, 6, dx=0.2, dz=0.02),
    "strips_sides": lambda: _cloud(9, 141, 31, dx=0.02, dz=0.09), "strips_by_x": lambda: _cloud(12, 150, 30, dx=0.02, dy=0.05, dz=0.05),
    "strips_by_y": lambda: _cloud(150, 12, 30, dx=0.05, dy=0.02, dz=0.05),
    # (1024 rows: a spacing whose multiples FP32 holds; at 0.1 the coordinates' rounding, half an ulp of 102.4
    # or 4e-5 of a cell, takes the planes to 6.5e-6 and the ring to 8.8e-6)
    "strips_1024_rows": lambda: _cloud(5, 1024, 2, dx=0.0625), "strips_l15": lambda: _cloud(70, 70, 61, dx=0.02, dz=0.02, nmu=12),
    "polarized": lambda: pol_blob(nmu=8, nphi=16),
}


@pytest.mark.parametrize("name", list(GRIDS))
def test_planes_match_point_order(name):
    w = GRIDS[name]()
    a, b = S.make_rte(w), S.make_rte(w)
    b.set_option("sweep_ring", 0)
    for r in (a, b):
        r.solve(3, verbose=False)
    assert a.timing("sweep_planes") == 1.0 and b.timing("sweep_planes") == 0.0
    for k in ("do_radiance", "do_source", "source"):
        x, y = a.state_array(k), b.state_array(k)
        if w.nstokes == 1:
            x, y = [x], [y]
        for i in range(len(x)):
            assert rel_l2(x[i], y[i]) < 2e-6, (k, i)


def test_grids_the_planes_do_not_take_keep_their_sweep():
    """Ordinates that go by z in thin layers and by a side in thick ones take
    the ring, as do strips of one long line, and periodic grids the point
    order; all are what they were."""
    w = _cloud(7, 8, 9, dx=0.05, z=0.4 + 0.9 * (np.arange(9) / 8.0) ** 2.5)
    a, b = S.make_rte(w), S.make_rte(w)
    b.set_option("sweep_ring", 0)
    for r in (a, b):
        r.solve(3, verbose=False)
    assert a.timing("sweep_planes") == 0.0 and a.timing("sweep_ring") == 1.0
    assert rel_l2(a.state_array("do_radiance"), b.state_array("do_radiance")) < 2e-6
    d = S.make_rte(_cloud(4, 1100, 3, dx=0.3, dz=0.03))
    d.solve(1, verbose=False)
    assert d.timing("sweep_planes") == 0.0 and d.timing("sweep_ring") == 1.0
    w.bc = "periodic"
    c = S.make_rte(w)
    c.solve(2, verbose=False)
    assert c.timing("sweep_planes") == 0.0 and c.timing("sweep_ring") == 0.0


def test_grids_past_the_ring_keep_their_fp64_steps():
    """A grid whose ring does not fit in LDS sweeps point by point in FP64, also
    where strips of planes would fit: bit for bit the point-ordered sweep."""
    rng = np.random.default_rng(3)
    shape = (111, 109, 110)
    ext = rng.lognormal(0.0, 0.5, shape).astype(np.float32)
    w = S.Workload("past_ring", 0.05, 0.05, (0.04 * np.arange(110)).astype(np.float32),
                   [(ext, np.full(shape, 0.95, np.float32), S.hg_legendre(0.5, 8))], bc="open", nmu=2, nphi=4)
    a, b = (S.make_rte(w, max_total_mb=50000.0, adapt_grid_factor=1.0) for _ in range(2))
    b.set_option("sweep_ring", 0)
    for r in (a, b):
        r.solve(2, verbose=False)
    assert a.timing("sweep_planes") == 0.0 and a.timing("sweep_ring") == 0.0
    assert np.array_equal(a.state_array("do_radiance"), b.state_array("do_radiance"))


def test_do_source_follows_the_sweep_that_wrote_it():
    """Each sweep has its own order of the DO source rows; they read back by
    point whichever sweep ran last, also where a graph captured earlier is
    replayed after iterations launched one by one in another order."""
    w = _cloud(14, 11, 10, nmu=8)
    a = S.make_rte(w)
    got = []
    for ring, graph in ((1, 1), (0, 0), (1, 1), (2, 1), (1, 0), (2, 1), (1, 1), (0, 1), (1, 1)):
        a.set_option("sweep_ring", ring)
        a.set_option("iteration_graph", graph)
        a.solve(60, verbose=False)
        got.append(a.state_array("do_source"))
    for x in got[1:]:
        assert rel_l2(x, got[0]) < 5e-6


def test_options_switch_between_sweeps_on_one_state():
    """Planes, ring, point order and planes again on one state, iterations from
    graphs: each solve is the one a state of its own gives."""
    w = _cloud(14, 11, 10, nmu=8)
    a = S.make_rte(w)
    got = []
    for opt in (1, 2, 0, 1, 2):
        a.set_option("sweep_ring", opt)
        a.solve(60, verbose=False)
        assert a.timing("iteration_graph_active") == 1.0
        assert a.timing("sweep_planes") == (1.0 if opt == 1 else 0.0)
        got.append((a.num_iterations, a.state_array("source")))
    assert np.array_equal(got[0][1], got[3][1]) and np.array_equal(got[1][1], got[4][1])
    for n, s in got[1:]:
        assert n == got[0][0] and rel_l2(s, got[0][1]) < 5e-6
