"""The point-ordered sweep from per-ordinate records against the general trace
(every point traced again in every sweep, in the octant's levels): FP64 in
both, so radiances agree to FP32 rounding.  Sizes: the smallest grids, points
around the 64-record chunks and their multiples, rows of doubles and (above
20480 points) of floats, several cells per trace (periodic), refined cells."""
import numpy as np
import pytest

from at3d_amd import synthetic as S
from tests.scenes import pol_blob, rel_l2

pytestmark = [pytest.mark.gpu, pytest.mark.filterwarnings("ignore:solution did not converge")]


def _cloud(nx, ny, nz, bc="open", nmu=8, **kw):
    w = S.cloud_field(nx=nx, ny=ny, nz=nz, dx=0.05, dz=0.9 / (nz - 1), z0=0.4, seed=3, nmu=nmu, nphi=2 * nmu, **kw)
    w.bc = bc
    return w


@pytest.mark.parametrize("make", [
    lambda: _cloud(2, 2, 3), lambda: _cloud(4, 4, 5, "periodic"),
    lambda: _cloud(9, 7, 11), lambda: _cloud(9, 7, 11, "periodic"), lambda: _cloud(5, 13, 6, "periodic", nmu=16),
    lambda: _cloud(31, 30, 23), lambda: pol_blob(bc="periodic")],
    ids=["2x2x3", "4x4x5p", "9x7x11", "9x7x11p", "5x13x6p_l15", "31x30x23", "polarized_p"])
def test_records_match_general_trace(make):
    a, b = S.make_rte(make()), S.make_rte(make())
    a.set_option("sweep_ring", 0)
    b.set_option("sweep_general", 1)
    for r in (a, b):
        r.solve(3, verbose=False)
    # the same FP64 sums before the rounding to FP32: at most a last place of
    # a radiance now and then
    assert rel_l2(a.state_array("do_radiance"), b.state_array("do_radiance")) < 2e-7
    assert rel_l2(a.state_array("source"), b.state_array("source")) < 5e-7


def test_graph_replay_matches_host_iterations_and_repeats():
    """Iterations from captured graphs, several solves with other work between,
    against iterations launched by the host."""
    w = _cloud(7, 6, 9, "periodic")
    a, b = S.make_rte(w), S.make_rte(w)
    b.set_option("iteration_graph", 0)
    b.solve(40, verbose=False)
    for _ in range(3):
        a.solve(40, verbose=False)
        assert a.timing("iteration_graph_active") == 1
        assert a.num_iterations == b.num_iterations
        assert rel_l2(a.state_array("source"), b.state_array("source")) < 1e-6
        a.fluxes


def test_refined_grid_matches_general_trace():
    w = _cloud(9, 8, 9)
    a, b = S.make_rte(w, split_accuracy=0.03), S.make_rte(w, split_accuracy=0.03)
    b.set_option("sweep_general", 1)
    for r in (a, b):
        r.solve(40, verbose=False)
    assert a.state_size("npts") > a.plan_size("npts")
    assert a.state_size("npts") == b.state_size("npts") and a.num_iterations == b.num_iterations
    assert np.array_equal(a.grid_arrays()["gridptr"], b.grid_arrays()["gridptr"])
    assert rel_l2(a.state_array("source"), b.state_array("source")) < 2e-6
