"""Plans without an attenuation map on the row-lane kernels (no factors, every
e^{-A} = 1): projection, both backprojections and ordered-subset EM against the
oracle, at the edges of the column rounds and tiles and of the rows per lane."""
import numpy as np
import pytest

from conftest import report_parity
from niftyrec_amd import phantoms
from oracle import orc

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


@pytest.mark.parametrize("shape, V, K", [((1, 1, 1), 1, 0), ((17, 1, 17), 3, 3), ((64, 33, 64), 4, 5),
                                         ((65, 32, 65), 4, 7), ((129, 97, 129), 3, 21), ((192, 4, 192), 3, 11),
                                         ((30, 128, 30), 4, 0)])
def test_no_attenuation(shape, V, K):
    from niftyrec_amd.api import ADJOINT, Plan
    rng = np.random.default_rng(7)
    act = rng.random(shape, dtype=np.float32) + 0.1
    cams = rng.uniform(0, 2 * np.pi, V).astype(np.float32)
    psf = phantoms.gaussian_psf(shape[2], K, 0.5, 1.6) if K else None
    plan = Plan(shape, cams, psf)
    tag = "%dx%dx%d, %d views, K=%d, no attenuation" % (shape[2], shape[1], shape[0], V, K)
    report_parity("project (%s)" % tag, plan.project(_t(act)).cpu().numpy(), orc.project(act, None, cams, psf),
                  orc.project(act, None, cams, psf, dtype=np.float64))
    y = rng.random((V,) + shape[1:], dtype=np.float32)
    report_parity("backproject (%s)" % tag, plan.backproject(_t(y)).cpu().numpy(), orc.backproject(y, None, cams, psf),
                  orc.backproject(y, None, cams, psf, dtype=np.float64))
    report_parity("adjoint (%s)" % tag, plan.backproject(_t(y), mode=ADJOINT, truncate=False).cpu().numpy(),
                  orc.backproject(y, None, cams, psf, 0.0, 0.0, 0, mode=1),
                  orc.backproject(y, None, cams, psf, 0.0, 0.0, 0, mode=1, dtype=np.float64))
    x = _t(np.ones(shape))
    plan.osem(x, _t(y), subsets=1, iterations=1)
    one = np.ones(shape, np.float32)
    report_parity("em update (%s)" % tag, x.cpu().numpy(), orc.mlem_step(one, y, None, cams, psf),
                  orc.mlem_step(one, y, None, cams, psf, dtype=np.float64))
