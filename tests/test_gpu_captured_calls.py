"""Single operations and OSEM recorded into a HIP graph: every replay gives what
the call gives on a fresh plan at that moment, whatever other calls, maps and
activities the plan saw in between (the keys of the cached factors and forward
sums are compared on the device, and a graph's launch tables are its own)."""
import numpy as np
import pytest

from niftyrec_amd import phantoms

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("shape, K, V", [((33, 31, 33), 5, 6), ((72, 20, 72), 3, 5), ((72, 130, 72), 3, 3)])
def test_replays_follow_the_content(shape, K, V):
    from niftyrec_amd.api import ADJOINT, Plan
    gen = torch.Generator(device="cuda").manual_seed(9)
    rand = lambda *s: torch.rand(s, device="cuda", generator=gen)  # noqa: E731
    cams = np.linspace(0.1, 5.0, V).astype(np.float32)
    psf = phantoms.gaussian_psf(shape[2], K, 0.5, 1.6)
    A, B, S = rand(*shape), rand(*shape), rand(V, *shape[1:])
    M, N = 0.05 * rand(*shape), 0.05 * rand(*shape)
    X = torch.empty(shape, device="cuda")

    def osem(p):
        X.fill_(1.0)
        return p.osem(X, S, N, subsets=2)

    ops = [lambda p: p.project(A, M), lambda p: p.project(A), lambda p: p.backproject(S),
           lambda p: p.backproject(S, M, mode=ADJOINT, truncate=False),
           lambda p: p.gradient_attenuation(S, A, M, exact=True, truncate=False),
           lambda p: p.gradient_attenuation(S, A, M),
           lambda p: torch.cat([t.flatten() for t in p.project_backward(S, A, M)]), osem]
    others = [lambda p: p.project(B, N), lambda p: p.backproject(S, mode=ADJOINT), lambda p: p.project(B),
              lambda p: p.gradient_attenuation(S, B, M, exact=True)]
    cold = lambda p: p.backproject(S, truncate=False)  # noqa: E731  (first called under capture)
    plan = Plan(shape, cams, psf)
    plan.set_tuning(2, 0)  # (fixed chunks: a fresh plan's OSEM takes the same)

    def fresh(op):
        p = Plan(shape, cams, psf)
        p.set_tuning(2, 0)
        return op(p).clone()

    for op in ops + others + ops:
        op(plan)
    graphs = []
    ops.append(cold)
    for op in ops:
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            out = op(plan)
        graphs.append((g, out))
    for step in range(3):
        for k, (op, (g, out)) in enumerate(zip(ops, graphs)):
            ref = fresh(op)
            for twice in range(2):
                out.zero_()
                g.replay()
                torch.cuda.synchronize()
                assert torch.equal(out, ref), (step, k, twice)
            eager = op(plan)
            torch.cuda.synchronize()
            assert torch.equal(eager, ref), (step, k)
            other = others[(step + k) % len(others)]
            assert torch.equal(other(plan), fresh(other)), (step, k)
        A.mul_(0.9)
        M.mul_(0.8)
