"""Operations in batches of views against all views at once, a batch's sums added
to those of the batches before: rows of 2, 4, 6 and 8 per lane, a partly filled
one, a tall plan (two row halves); and both gradients at once against each
operation.  The sums of 7 views are of 7 terms in another order: their
difference is below 7 x 2^-24 of the sum of the terms' magnitudes, so below 1e-6
of the largest such sum."""
import numpy as np
import pytest

from niftyrec_amd import phantoms

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("shape, K", [((20, 30, 20), 3), ((33, 33, 33), 5), ((70, 96, 70), 7), ((24, 128, 24), 0),
                                      ((72, 140, 72), 3)])
@pytest.mark.parametrize("truncate", [False, True])
def test_batches_of_views(shape, K, truncate):
    from niftyrec_amd.api import ADJOINT, REFERENCE, Plan
    gen = torch.Generator(device="cuda").manual_seed(11)
    rand = lambda *s: torch.rand(s, device="cuda", generator=gen)  # noqa: E731
    V = 7
    act, mu, sino = rand(*shape), 0.05 * rand(*shape), rand(V, *shape[1:]) - 0.4
    plan = Plan(shape, np.linspace(0.1, 5.0, V).astype(np.float32),
                phantoms.gaussian_psf(shape[2], K, 0.5, 1.6) if K else None)
    ops = [lambda S, m=m, a=a: plan.backproject(S, a, mode=m, truncate=truncate)
           for m in (ADJOINT, REFERENCE) for a in (mu, None)]
    ops.append(lambda S: plan.gradient_attenuation(S, act, mu, exact=True, truncate=truncate))
    plan.set_tuning(0, V)
    ref = [op(sino) for op in ops]
    size = [op(sino.abs()) for op in ops[:4]] + [plan.gradient_attenuation(-sino.abs(), act, mu, exact=True)]
    for vb in (1, 3):
        plan.set_tuning(0, vb)
        got = [op(sino) for op in ops]
        for k, (g, r, m) in enumerate(zip(got, ref, size)):
            assert m.max() > 0 and (g - r).abs().max() <= 1e-6 * m.abs().max(), (k, vb)
        both = plan.project_backward(sino, act, mu, truncate=truncate)
        assert torch.equal(both[0], got[0]) and torch.equal(both[1], got[4])
