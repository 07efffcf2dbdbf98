"""The reference attenuation gradient of a created plan (row-lane kernels: a
projection without PSF for the chunk sums, the reverse sweep, the reference
pull) against the oracle: one plane to several chunks, one to three column
rounds, every number of rows per lane, view batches, truncation of signed
weights."""
import numpy as np
import pytest

from conftest import report_parity
from niftyrec_amd import phantoms
from oracle import orc

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


@pytest.mark.parametrize("shape, V, K, batch", [((1, 1, 1), 1, 0, 0), ((17, 3, 17), 3, 3, 0), ((64, 33, 64), 4, 7, 0),
                                                ((65, 64, 65), 5, 5, 2), ((129, 97, 129), 2, 21, 0),
                                                ((40, 20, 40), 6, 0, 4)])
def test_reference_gradient(shape, V, K, batch):
    from niftyrec_amd.api import Plan
    rng = np.random.default_rng(17)
    act = rng.random(shape, dtype=np.float32) + 0.1
    mu = (0.05 * rng.random(shape, dtype=np.float32)).astype(np.float32)
    cams = rng.uniform(0, 2 * np.pi, V).astype(np.float32)
    psf = phantoms.gaussian_psf(shape[2], K, 0.5, 1.6) if K else None
    y = rng.random((V,) + shape[1:], dtype=np.float32)
    plan = Plan(shape, cams, psf)
    plan.set_tuning(0, batch)
    g = plan.gradient_attenuation(_t(y), _t(act), _t(mu)).cpu().numpy()
    report_parity("plan reference gradient %s, %d views, K=%d, batch %d" % (shape, V, K, batch), g,
                  orc.gradient_ref(y, act, mu, cams, psf), orc.gradient_ref(y, act, mu, cams, psf, dtype=np.float64))
    s = y.copy()
    s[::2] *= -1.0  # whole views negative: where they dominate, the result is truncated
    g = plan.gradient_attenuation(_t(s), _t(act), _t(mu)).cpu().numpy()
    assert (g >= 0).all()
    r = orc.gradient_ref(s, act, mu, cams, psf, dtype=np.float64)
    assert np.abs(g - r).max() <= 1e-4 * max(np.abs(orc.gradient_ref(y, act, mu, cams, psf)).max(), 1e-30)
