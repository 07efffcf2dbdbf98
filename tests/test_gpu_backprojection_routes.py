"""Backprojections without attenuation of wide and tall plans, which take the
sweep kernels or the tile kernels by the work of either, in turn on one plan with
those that take the others' volumes (attenuation, the adjoint, the gradients, OSEM),
against the oracle: the two kinds of rotated-frame volumes do not meet."""
import numpy as np
import pytest

from conftest import report_parity
from niftyrec_amd import phantoms
from oracle import orc

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("shape, V, K", [((72, 130, 72), 3, 21), ((200, 40, 200), 2, 21), ((68, 250, 68), 2, 5)])
def test_routes_in_turn(shape, V, K):
    from niftyrec_amd.api import ADJOINT, REFERENCE, Plan
    rng = np.random.default_rng(17)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()  # noqa: E731
    act = rng.random(shape, dtype=np.float32)
    mu = (4.0 / shape[0] * rng.random(shape, dtype=np.float32)).astype(np.float32)
    cams = rng.uniform(0, 2 * np.pi, V).astype(np.float32)
    psf = phantoms.gaussian_psf(shape[2], K, 0.5, 1.6)
    y = rng.random((V,) + shape[1:], dtype=np.float32)
    A, M, Y = t(act), t(mu), t(y)
    ref = {(m, mode): [orc.backproject(y, mu if m else None, cams, psf, 0.0, 0.0, 0, mode=mode, dtype=d)
                       for d in (np.float32, np.float64)] for m in (False, True) for mode in (0, 1)}
    plan = Plan(shape, cams, psf)

    def check(m, mode):
        b = plan.backproject(Y, M if m else None, mode=ADJOINT if mode else REFERENCE, truncate=False)
        report_parity("backproject (%dx%d, K=%d, mu=%s, adjoint=%s)" % (shape[2], shape[1], K, m, bool(mode)),
                      b.cpu().numpy(), *ref[m, mode])

    for between in (None, lambda: plan.osem(torch.ones_like(A), Y, M, subsets=1), lambda: plan.project(A),
                    lambda: plan.gradient_attenuation(Y, A, M), lambda: plan.project_backward(Y, A, M)):
        if between is not None:
            between()
        for m, mode in ((False, 0), (True, 0), (False, 1), (True, 1), (False, 0)):
            check(m, mode)
