"""The direct-beam term of the gradient, summed over sun paths traced on the
device, against the Jacobian of the same call, whose direct-beam part comes
from the host's stored paths: sum over pixels of U (R - M) J is the gradient
(both FP64 sums of the same terms; J is rounded to FP32, 6e-8 a term).  Suns
overhead (every bottom point's path is a longest one, so it takes the next
point's too), oblique and low, open and periodic, odd sizes."""
import numpy as np
import pytest

from at3d_amd import gradient as G
from at3d_amd import synthetic as S
from tests.scenes import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bc", ["open", "periodic"])
@pytest.mark.parametrize("mu,az", [(-1.0, 0.0), (-0.5, 0.0), (-0.6, 37.0), (-0.2, 200.0)])
def test_gradient_is_the_jacobian_contracted(bc, mu, az):
    rng = np.random.default_rng(4)
    shape = (7, 5, 6)
    ext = rng.uniform(0.1, 4.0, shape).astype(np.float32)
    alb = rng.uniform(0.6, 1.0, shape).astype(np.float32)
    w = S.Workload("thin", 0.1, 0.1, np.linspace(0, 0.6, 6).astype(np.float32), [(ext, alb, S.hg_legendre(0.7, 16))],
                   bc=bc, nmu=4, nphi=8, solarmu=mu, solaraz_deg=az, solacc=1e-4)
    rte = S.make_rte(w)
    rte.solve(100, verbose=False)
    rays = S.view_rays(w, [(0.0, 0.0), (40.0, 30.0)], 9, 8)
    n = rays["ray_x"].size
    meas = rng.uniform(0.02, 0.2, n).astype(np.float32)
    sp = list(rte.medium)[0]
    idx = tuple(a.ravel() for a in np.indices(shape))
    g, _, out, jac = G.levis_approximation_grad(rte, dict(rays, measurement_data=meas),
                                                [(sp, "extinction"), (sp, "ssalb")], indices_for_jacobian=idx)
    res = out["I"].astype(np.float64) - meas
    back = np.einsum("dgp,p->dg", jac[0].astype(np.float64), res)
    for d in range(2):
        assert rel_l2(g[d].ravel(), back[d]) < 2e-6
