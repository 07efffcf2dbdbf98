"""The general path (cameras about three axes, backgrounds, a PSF wider than
the sweeps take) in batches of views: one view, a batch that does not divide
the view count, and all views at once, with and without depth chunks, against
the oracle."""
import numpy as np
import pytest

from conftest import report_parity
from niftyrec_amd import phantoms
from oracle import orc

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


@pytest.mark.parametrize("batch, chunks", [(1, 0), (3, 0), (0, 0), (3, 1), (2, 5)])
@pytest.mark.parametrize("shape, K, bg", [((18, 21, 18), 5, 0.0), ((26, 9, 26), 23, 0.0), ((12, 17, 12), 0, 0.3),
                                          ((10, 70, 10), 3, 0.0)])
def test_general_path_in_batches(shape, K, bg, batch, chunks):
    from niftyrec_amd.api import Plan
    rng = np.random.default_rng(11)
    act = rng.random(shape, dtype=np.float32) + 0.1
    mu = 0.05 * rng.random(shape, dtype=np.float32)
    cams = rng.uniform(-0.5, 0.5, (3, 5)).astype(np.float32)
    psf = phantoms.gaussian_psf(shape[2], K, 0.6, 2.0) if K else None
    plan = Plan(shape, cams, psf, background=bg)
    plan.set_tuning(chunks, batch)
    tag = "general %s, K=%d, bg=%g, batch %d, chunks %d" % (shape, K, bg, batch, chunks)
    report_parity("project " + tag, plan.project(_t(act), _t(mu)).cpu().numpy(), orc.project(act, mu, cams, psf, bg),
                  orc.project(act, mu, cams, psf, bg, dtype=np.float64))
    y = rng.random((5,) + shape[1:], dtype=np.float32)
    report_parity("backproject " + tag, plan.backproject(_t(y), _t(mu)).cpu().numpy(),
                  orc.backproject(y, mu, cams, psf, bg), orc.backproject(y, mu, cams, psf, bg, dtype=np.float64))
    report_parity("gradient " + tag, plan.gradient_attenuation(_t(y), _t(act), _t(mu)).cpu().numpy(),
                  orc.gradient_ref(y, act, mu, cams, psf, bg), orc.gradient_ref(y, act, mu, cams, psf, bg, dtype=np.float64))
