"""Wide (more than 192 columns) and tall (more than 128 rows) plans on the tile
kernels: projection, both backprojections, the exact gradients and ordered
subsets against the oracle, at the edges of the tiles, of the rows a column's
lanes hold and of the halo (the permutes across a column's lanes), with and
without attenuation; and the sizes whose OSEM the sweep kernels keep (0 tiles)."""
import numpy as np
import pytest

from conftest import report_parity
from niftyrec_amd import phantoms
from oracle import orc

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


@pytest.mark.parametrize("shape, V, K, attenuated, tiles", [
    ((65, 129, 65), 3, 21, True, 0), ((70, 192, 70), 3, 7, True, 2), ((66, 193, 66), 2, 0, True, 0),
    ((129, 256, 129), 2, 17, True, 3), ((72, 168, 72), 3, 19, False, 2), ((72, 167, 72), 3, 19, False, 0), ((193, 17, 193), 2, 21, True, 4),
    ((200, 33, 200), 2, 0, False, 4), ((257, 65, 257), 2, 5, True, 5), ((194, 128, 194), 2, 11, True, 4),
    ((64, 129, 64), 2, 5, True, 0), ((200, 16, 200), 2, 3, True, 0), ((70, 257, 70), 2, 3, True, 0)])
def test_wide_and_tall_plans(shape, V, K, attenuated, tiles):
    from niftyrec_amd.api import ADJOINT, Plan
    rng = np.random.default_rng(31)
    act = rng.random(shape, dtype=np.float32) + 0.1
    mu = (4.0 / shape[0] * rng.random(shape, dtype=np.float32)).astype(np.float32) if attenuated else None
    cams = rng.uniform(0, 2 * np.pi, V).astype(np.float32)
    psf = phantoms.gaussian_psf(shape[2], K, 0.5, 1.6) if K else None
    if psf is not None:
        psf[:, :, 0] *= 1.2  # asymmetric: correlation differs from convolution
    plan = Plan(shape, cams, psf)
    M = None if mu is None else _t(mu)
    tag = "(%dx%dx%d, %d views, K=%d, mu=%s)" % (shape[2], shape[1], shape[0], V, K, attenuated)
    y = rng.random((V,) + shape[1:], dtype=np.float32)
    x = _t(np.ones(shape))
    plan.osem(x, _t(y), M, subsets=1, iterations=1)
    assert plan.projector() == tiles
    one = np.ones(shape, np.float32)
    report_parity("em update " + tag, x.cpu().numpy(), orc.mlem_step(one, y, mu, cams, psf),
                  orc.mlem_step(one, y, mu, cams, psf, dtype=np.float64))
    report_parity("project " + tag, plan.project(_t(act), M).cpu().numpy(), orc.project(act, mu, cams, psf),
                  orc.project(act, mu, cams, psf, dtype=np.float64))
    report_parity("backproject " + tag, plan.backproject(_t(y), M).cpu().numpy(), orc.backproject(y, mu, cams, psf),
                  orc.backproject(y, mu, cams, psf, dtype=np.float64))
    adj = (orc.backproject(y, mu, cams, psf, 0.0, 0.0, 0, mode=1),
           orc.backproject(y, mu, cams, psf, 0.0, 0.0, 0, mode=1, dtype=np.float64))
    report_parity("adjoint " + tag, plan.backproject(_t(y), M, mode=ADJOINT, truncate=False).cpu().numpy(), *adj)
    if mu is None:
        return
    grad = (orc.gradient_mu(y, act, mu, cams, psf, dtype=np.float32), orc.gradient_mu(y, act, mu, cams, psf, dtype=np.float64))
    ga, gm = plan.project_backward(_t(y), _t(act), M)
    report_parity("backward, activity " + tag, ga.cpu().numpy(), *adj)
    report_parity("backward, attenuation " + tag, gm.cpu().numpy(), *grad)
    plan.set_tuning(0, 1)  # gradient in one-view batches, from the sums already there
    g = plan.gradient_attenuation(_t(y), _t(act), M, exact=True, truncate=False).cpu().numpy()
    report_parity("gradient " + tag, g, *grad)
    ref = plan.gradient_attenuation(_t(y), _t(act), M).cpu().numpy()
    report_parity("reference gradient " + tag, ref, orc.gradient_ref(y, act, mu, cams, psf),
                  orc.gradient_ref(y, act, mu, cams, psf, dtype=np.float64))


def test_osem_with_maps_that_change():
    """The structural OSEM data (chunking, launch table) outlive the map, the
    factors and sensitivities follow it: passes over two maps, a single
    operation with the other map in between, another epsilon, then the first
    map again, each bit-identical to a fresh plan's with the same chunking."""
    from niftyrec_amd.api import Plan
    shape, V = (72, 180, 72), 6
    gen = torch.Generator(device="cuda").manual_seed(9)
    rand = lambda *s: torch.rand(s, device="cuda", generator=gen)  # noqa: E731
    cams = np.linspace(0, 5, V).astype(np.float32)
    psf = phantoms.gaussian_psf(shape[2], 7, 0.5, 1.6)
    Y, M = rand(V, *shape[1:]) + 0.1, [0.05 * rand(*shape) for _ in range(2)]
    M.append(None)

    def run(plan, m, eps):
        x = torch.ones(shape, device="cuda")
        return plan.osem(x, Y, M[m], subsets=3, iterations=2, epsilon=eps)

    def fresh():
        p = Plan(shape, cams, psf)
        p.set_tuning(5, 0)
        return p

    plan = fresh()
    for m, eps, between in [(0, 1e-6, None), (1, 1e-6, None), (1, 1e-6, 0), (1, 1e-3, None), (0, 1e-3, 1), (2, 1e-3, 0),
                            (0, 1e-6, None)]:
        if between is not None:
            plan.backproject(Y, M[between])
        assert torch.equal(run(plan, m, eps), run(fresh(), m, eps)), (m, eps, between)
