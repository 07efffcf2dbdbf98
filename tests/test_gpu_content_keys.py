"""The single operations' content keys, compared on the device: whatever ran
before on the plan (other activities, other maps, a map rewritten in place, no
map, an invalidation), an operation's result is bit-identical to a fresh
plan's.  Sizes at the edges of the packed 32 x 32 tiles and of the planes one
block packs."""
import numpy as np
import pytest

from niftyrec_amd import phantoms

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("shape, K", [((1, 1, 1), 0), ((33, 31, 33), 5), ((65, 40, 65), 3), ((180, 2, 180), 7)])
def test_keys_follow_the_content(shape, K):
    from niftyrec_amd.api import ADJOINT, Plan
    gen = torch.Generator(device="cuda").manual_seed(5)
    rand = lambda *s: torch.rand(s, device="cuda", generator=gen)  # noqa: E731
    cams = np.linspace(0.1, 5.0, 4).astype(np.float32)
    psf = phantoms.gaussian_psf(shape[2], K, 0.5, 1.6) if K else None
    A = [rand(*shape) for _ in range(2)]
    M = [0.05 * rand(*shape) for _ in range(2)]
    S = rand(4, *shape[1:])

    def fresh():
        return Plan(shape, cams, psf)

    ops = {"project": lambda p, a, m: p.project(a, m),
           "adjoint": lambda p, a, m: p.backproject(S, m, mode=ADJOINT, truncate=False),
           "gradient": lambda p, a, m: p.gradient_attenuation(S, a, m, exact=True, truncate=False),
           "backward": lambda p, a, m: torch.cat([t.flatten() for t in p.project_backward(S, a, m)]),
           "bare": lambda p, a, m: p.project(a)}
    plan = fresh()
    steps = [("project", 0, 0), ("gradient", 0, 0), ("project", 1, 0), ("gradient", 0, 0), ("backward", 0, 0),
             ("adjoint", 0, 1), ("gradient", 0, 0), ("backward", 1, 1), ("bare", 1, 0), ("gradient", 1, 1),
             ("backward", 1, 1), ("rewrite", 0, 1), ("project", 1, 1), ("adjoint", 0, 1), ("rewrite", 0, 1),
             ("gradient", 1, 1), ("invalidate", 0, 0), ("backward", 1, 1), ("backward", 0, 0)]
    for k, (op, a, m) in enumerate(steps):
        if op == "rewrite":
            M[m].mul_(0.75)
        elif op == "invalidate":
            plan.invalidate()
        else:
            got, ref = ops[op](plan, A[a], M[m]), ops[op](fresh(), A[a], M[m])
            assert torch.equal(got, ref), (k, op, a, m)
