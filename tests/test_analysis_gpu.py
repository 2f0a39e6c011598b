"""DO->SH by azimuth and Legendre sums against the product with the dense tables
in FP64.  A coefficient is at most 19 + 16 products of FP32 factors, each rounded
on the way: 38 half ulps of its terms' sizes at worst, 2.3e-6, and the square
root of that when they add at random, 4e-7.  The dense product that serves larger
sets sums NANG, 448 at NMU 18: 1.3e-6 at random.  Angle sets from one zenith pair to
the largest the kernel takes (odd and even azimuth counts, M below L) and one
past it, tiles that are full, ragged and fewer than the workgroups."""
import numpy as np
import pytest

from at3d_amd import synthetic as S
from tests.scenes import pol_blob, rel_l2

pytestmark = [pytest.mark.gpu, pytest.mark.filterwarnings("ignore:solution did not converge")]


def _cloud(nx, ny, nz, nmu, nphi):
    return S.cloud_field(nx=nx, ny=ny, nz=nz, dx=0.05, dz=0.05, z0=0.4, nmu=nmu, nphi=nphi)


@pytest.mark.parametrize("nmu,nphi,shape", [(2, 4, (5, 4, 3)), (4, 8, (8, 8, 8)), (6, 12, (9, 7, 5)), (8, 16, (13, 11, 9)),
                                            (8, 8, (4, 4, 4)), (10, 18, (9, 8, 7)), (12, 24, (16, 12, 11)),
                                            (14, 28, (7, 9, 6)), (16, 24, (9, 8, 7)), (16, 32, (33, 20, 11)),
                                            (18, 36, (9, 8, 7))])
def test_radiances_match_the_dense_product(nmu, nphi, shape):
    w = _cloud(*shape, nmu, nphi)
    a = S.make_rte(w)
    a.solve(3, verbose=False)
    ref = a.state_array("do_radiance").astype(np.float64).T @ a.plan_array("wmat").astype(np.float64)
    r = a.state_array("radiance")
    kept = np.arange(r.shape[1]) < a.state_array("nr")[:, None]
    assert np.all(r[~kept] == 0.0)
    assert rel_l2(r[kept], ref[kept]) < (5e-7 if nmu <= 16 else 1.3e-6)


@pytest.mark.parametrize("nmu,nphi", [(4, 8), (8, 16), (12, 24), (16, 24), (16, 32)])
def test_polarized_matches_the_dense_product(nmu, nphi):
    """All three components, and the rows' zeros, through a solve (the dense
    kernel's own error is the larger: sums of NANG terms)."""
    w = pol_blob(nmu=nmu, nphi=nphi)
    a, b = S.make_rte(w), S.make_rte(w)
    b.set_option("dense_analysis", 1)
    for r in (a, b):
        r.solve(8, verbose=False)
    for k in ("radiance", "source"):
        for x, y in zip(a.state_array(k), b.state_array(k)):
            assert rel_l2(x, y) < 2e-6
    # (a row's extent may differ by the terms at its truncation's threshold)
    n = np.arange(a.state_array("radiance").shape[2])
    for x in a.state_array("radiance"):
        assert np.all(x[n[None, :] >= a.state_array("nr")[:, None]] == 0.0)


def test_rows_stay_zero_past_their_counts():
    """Rows written by one path and then another: solves from graphs and one by
    one, again on the same state and after the dense product, each with the
    bytes a new state gives."""
    w = _cloud(14, 11, 10, 8, 16)
    want = []
    for graph in (0, 1):   # (the acceleration's parameters come from the host or the device)
        r = S.make_rte(w)
        r.set_option("iteration_graph", graph)
        r.solve(60, verbose=False)
        want.append(r.state_array("radiance"))

    def past(r):
        x = r.state_array("radiance")
        return np.count_nonzero(x[np.arange(x.shape[1]) >= r.state_array("nr")[:, None]])
    a = S.make_rte(w)
    for dense, graph in ((0, 0), (1, 0), (0, 1), (0, 0), (1, 1), (0, 1)):
        a.set_option("dense_analysis", dense)
        a.set_option("iteration_graph", graph)
        a.solve(60, verbose=False)
        assert past(a) == 0
        if dense:
            assert rel_l2(a.state_array("radiance"), want[graph]) < 5e-6
        else:
            assert np.array_equal(a.state_array("radiance"), want[graph])
