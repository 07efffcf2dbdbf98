"""The work that programs have this library do, as cases that can be timed.

Every case goes through the public Python entry points: `niftyrec_amd.api.Plan`
and `Batch` on device tensors, `niftyrec_amd.torch_ops` for autograd, and the
array interface on host arrays.  Volumes are (nz, ny, nx) with y the rotation
axis, nz == nx; the sizes span the 32^3 check volume to the 256^3 x 180 view,
21 x 21 PSF joint reconstruction.

A case is a dict of plain values:
    op          project | backproject | gradient | autograd | osem | joint |
                batch | mlem_step
    n, ny       columns (x and z) and axial rows
    views       cameras
    psf         PSF size (odd), 0: none
    mu          attenuation map or not
    tilt        cameras about all three axes (off the axial fast path)
    adjoint     backproject: the exact adjoint instead of the reference pull
    subsets     osem, joint, batch: ordered subsets; mlem_step has none
    iterations  osem, batch: passes over the subsets
    problems    batch: number of problems (their sizes follow from `pick`)

`exact` evaluates the same operation in double precision with plain torch:
rotated volumes by bilinear (trilinear when tilted) row gathers, the separable
PSF as banded matrix products, attenuation as a cumulative sum along depth.
"""
import math
import random

import numpy as np
import torch

from niftyrec_amd import api
from niftyrec_amd.torch_ops import poisson_nll, project

BATCH_SHAPES = [(64, 64), (96, 96), (128, 128), (160, 96)]  # (n, ny) of the batched reconstructions
EPS = 1e-6


# ---- the cases -----------------------------------------------------------------

def listed():
    return [
        # a quick look at a small phantom: latency and launch counts
        dict(name="project_32", op="project", n=32, ny=24, views=16, psf=5, mu=True),
        # data simulation without attenuation, the 64^3 study size
        dict(name="project_64_nomu", op="project", n=64, ny=64, views=64, psf=7, mu=False),
        # clinical-size simulation with resolution model and attenuation
        dict(name="project_128", op="project", n=128, ny=128, views=120, psf=11, mu=True),
        # one backprojection, no attenuation correction (a user's own update rule around it)
        dict(name="backproject_128_nomu", op="backproject", n=128, ny=128, views=120, psf=11, mu=False,
             adjoint=False),
        # the reference library's attenuation gradient
        dict(name="gradient_64", op="gradient", n=64, ny=64, views=64, psf=7, mu=True),
        # the differentiable projector inside a training step: loss and both gradients
        dict(name="autograd_128", op="autograd", n=128, ny=128, views=120, psf=11, mu=True),
        # the headline reconstruction: ordered subsets with PSF and attenuation
        dict(name="osem_128", op="osem", n=128, ny=128, views=120, psf=11, mu=True, subsets=8, iterations=2),
        # a wide, short, odd-sized field of view without attenuation
        dict(name="osem_130x24_nomu", op="osem", n=130, ny=24, views=90, psf=11, mu=False, subsets=6, iterations=2),
        # many uneven reconstructions at once
        dict(name="batch_8", op="batch", problems=8, pick=3, subsets=8, iterations=1),
        # joint activity and attenuation estimation at full size: two alternations
        dict(name="joint_256", op="joint", n=256, ny=256, views=180, psf=21, mu=True, subsets=10),
        # the array interface on host arrays, one update per call, as existing scripts use it
        dict(name="mlem_step_host_96", op="mlem_step", n=96, ny=96, views=60, psf=11, mu=True),
        # cameras about three axes: the general rotation path
        dict(name="project_tilted_64", op="project", n=64, ny=64, views=32, psf=7, mu=True, tilt=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges."""
    op = rng.choice(["project", "project", "backproject", "backproject", "osem", "osem", "autograd", "gradient",
                     "joint", "batch", "mlem_step", "tilted"])
    if op == "batch":
        return dict(op="batch", problems=rng.randint(2, 8), pick=rng.randrange(10 ** 6), subsets=rng.choice([4, 6, 8]),
                    iterations=1)
    hi = dict(mlem_step=112, tilted=72, gradient=144, joint=192).get(op, 256)
    n, ny = _log_int(rng, 24, hi), _log_int(rng, 16, hi)
    views = _log_int(rng, 12, 32 if op == "tilted" else 180)
    psf = rng.choice([k for k in (0, 3, 5, 7, 11, 15, 21) if k < n // 2])
    mu = op in ("autograd", "gradient", "joint") or rng.random() < 0.6
    case = dict(op="project" if op == "tilted" else op, n=n, ny=ny, views=views, psf=psf, mu=mu)
    if op == "tilted":
        case["tilt"] = True
    if op == "backproject":
        case["adjoint"] = rng.random() < 0.5
    if op in ("osem", "joint"):
        case["subsets"] = rng.choice([s for s in (1, 4, 6, 8, 10) if s <= views // 3])
    if op == "osem":
        case["iterations"] = rng.randint(1, 3)
    return case


# ---- inputs --------------------------------------------------------------------

def _psf(n, K):
    """(n, K, K) Gaussians whose width grows with depth."""
    if not K:
        return None
    s0, s1 = 0.5 + 0.015 * K, 0.215 * K + 0.05
    t = np.arange(K) - (K - 1) / 2.0
    out = np.empty((n, K, K))
    for d in range(n):
        g = np.exp(-0.5 * (t / (s0 + (s1 - s0) * d / max(n - 1, 1))) ** 2)
        out[d] = np.outer(g, g)
        out[d] /= out[d].sum()
    return out.astype(np.float32)


def _cameras(views, tilt):
    a = (2 * np.pi * np.arange(views) / views).astype(np.float32)
    if not tilt:
        return a
    return np.stack([np.full(views, 0.12, np.float32), a, np.full(views, -0.07, np.float32)])


def _phantom(n, ny, rng, dev):
    """Ellipsoid body with random hot lesions, and its attenuation (a lung-like
    and a bone-like inclusion), float32 on the device."""
    z = torch.arange(n, device=dev, dtype=torch.float32).view(-1, 1, 1)
    y = torch.arange(ny, device=dev, dtype=torch.float32).view(1, -1, 1)
    x = torch.arange(n, device=dev, dtype=torch.float32).view(1, 1, -1)
    c, cy = (n - 1) / 2.0, (ny - 1) / 2.0
    ax, ay = 0.4375 * n, 0.42 * ny

    def ellipsoid(cx, cyy, cz, rx, ry, rz):
        return ((x - cx) / rx) ** 2 + ((y - cyy) / ry) ** 2 + ((z - cz) / rz) ** 2 <= 1.0

    body = ellipsoid(c, cy, c, ax, ay, ax)
    act = body.float()
    for _ in range(12):
        p = rng.uniform(-0.55, 0.55, 3)
        r = rng.uniform(0.03, 0.11, 3) * n + 0.6
        act += float(rng.uniform(2, 10)) * ellipsoid(c + p[0] * ax, cy + p[1] * ay, c + p[2] * ax, *map(float, r))
    scale = 20.0 / n  # the body's total attenuation does not depend on the sampling
    mu = body.float() * (0.15 * scale)
    mu[ellipsoid(c + 0.35 * ax, cy, c, 0.13 * n, 0.19 * ny, 0.16 * n) & body] = 0.05 * scale
    mu[ellipsoid(c - 0.4 * ax, cy, c + 0.3 * ax, 0.05 * n, 0.16 * ny, 0.05 * n) & body] = 0.30 * scale
    return act.contiguous(), mu.contiguous()


def _counts(act, mu, cams, total, gen):
    """Poisson counts of a plain (unblurred) projection scaled to `total`."""
    g = _Exact(act.shape[0], act.shape[1], cams, None, torch.float32, act.device)
    p = g.project(act, mu).clamp_min(0)
    return torch.poisson(p * (total / p.sum().clamp_min(1e-30)), generator=gen).contiguous()


def _batch_problem(pick, i):
    r = random.Random(pick * 1000 + i)
    n, ny = r.choice(BATCH_SHAPES)
    return dict(n=n, ny=ny, views=r.randint(60, 180), psf=r.choice([7, 11, 15]))


def _problem(c, seed, dev):
    """Inputs of a case: dict of activity, mu, counts, cameras, psf."""
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=dev).manual_seed(int(seed))
    n, ny = c["n"], c["ny"]
    act, mu = _phantom(n, ny, rng, dev)
    cams = _cameras(c["views"], c.get("tilt", False))
    if not c.get("mu", True):
        mu = None
    w = dict(activity=act, mu=mu, cameras=cams, psf=_psf(n, c["psf"]))
    if c.get("op") in ("osem", "joint", "mlem_step", "autograd", None):
        w["counts"] = _counts(act, mu, cams, 2.5 * c["views"] * n * ny, gen)
    elif c["op"] in ("backproject", "gradient"):  # what an update rule feeds back: noisy ratios about 1
        w["weights"] = 1.0 + 0.3 * torch.randn((c["views"], ny, n), device=dev, generator=gen)
    return w


def prepare(case, seed):
    dev = torch.device("cuda:0")
    op = case["op"]
    s = {"op": op, "case": case}
    if op == "batch":
        ps = [_problem(_batch_problem(case["pick"], i), 100 * seed + i, dev) for i in range(case["problems"])]
        plans = [api.Plan(tuple(p["activity"].shape), p["cameras"], p["psf"]) for p in ps]
        s.update(plans=plans, batch=api.Batch(plans), counts=[p["counts"] for p in ps], mu=[p["mu"] for p in ps])
        return s
    w = _problem(case, seed, dev)
    if op == "mlem_step":
        host = lambda t: None if t is None else t.cpu().numpy()  # noqa: E731
        s.update(activity=np.ones((case["n"], case["ny"], case["n"]), np.float32), counts=host(w["counts"]),
                 mu=host(w["mu"]), cameras=w["cameras"], psf=w["psf"])
        return s
    s["plan"] = api.Plan((case["n"], case["ny"], case["n"]), w["cameras"], w["psf"])
    if op == "autograd":  # an estimate on its way to the truth
        w["activity"] = (w["activity"] * 0.9 + 0.05).requires_grad_(True)
        w["mu"] = (w["mu"] * 0.8).requires_grad_(True)
    if op == "joint":
        w["mu"] = w["mu"] * 0.8
        s["plan"].set_tuning(16, 0)
    s.update((k, w[k]) for k in ("activity", "mu", "counts", "weights") if k in w)
    return s


def run(state):
    op, c = state["op"], state["case"]
    if op == "project":
        return state["plan"].project(state["activity"], state["mu"])
    if op == "backproject":
        return state["plan"].backproject(state["weights"], state["mu"],
                                         mode=api.ADJOINT if c["adjoint"] else api.REFERENCE)
    if op == "gradient":
        return state["plan"].gradient_attenuation(state["weights"], state["activity"], state["mu"])
    if op == "autograd":
        a, m = state["activity"], state["mu"]
        a.grad = m.grad = None
        loss = poisson_nll(project(a, m, state["plan"]), state["counts"])
        loss.backward()
        return loss, a.grad, m.grad
    if op == "osem":
        x = torch.ones_like(state["activity"])
        return state["plan"].osem(x, state["counts"], state["mu"], subsets=c["subsets"], iterations=c["iterations"],
                                  epsilon=EPS)
    if op == "batch":
        x = [torch.ones(p.shape, device="cuda:0") for p in state["plans"]]
        return state["batch"].osem(x, state["counts"], state["mu"], subsets=c["subsets"],
                                   iterations=c["iterations"], epsilon=EPS)
    if op == "joint":
        # alternate: one OSEM pass on the activity, one projected gradient step on mu
        plan, y = state["plan"], state["counts"]
        x = torch.ones_like(state["activity"])
        mu = state["mu"].clone()
        for _ in range(2):
            plan.osem(x, y, mu, subsets=c["subsets"], iterations=1, epsilon=EPS)
            m = mu.clone().requires_grad_(True)
            poisson_nll(project(x, m, plan), y).backward()
            with torch.no_grad():
                mu.sub_(0.01 * m.grad / m.grad.abs().max().clamp_min(1e-30)).clamp_(min=0.0)
        return x, mu, m.grad
    if op == "mlem_step":
        return api.mlem_step(state["activity"], state["counts"], state["cameras"], state["psf"], state["mu"],
                             epsilon=EPS)
    raise ValueError(op)


def work(case):
    """Inputs read once, outputs written once; per voxel and view a bilinear
    sample (7, also of mu), the separable PSF (4 psf), attenuation and sum (4)."""
    op = case["op"]
    if op == "batch":
        ws = [work(dict(_batch_problem(case["pick"], i), op="osem", mu=True, subsets=case["subsets"],
                        iterations=case["iterations"])) for i in range(case["problems"])]
        return {k: sum(w[k] for w in ws) for k in ("bytes", "flops")}
    n, P, V = case["n"] ** 2 * case["ny"], case["n"] * case["ny"], case["views"]
    m = 1 if case["mu"] else 0
    sweep = V * n * (7.0 + 4.0 * case["psf"] + (11.0 if m else 1.0))
    sino = 4.0 * V * P
    if op in ("project", "backproject"):
        return {"bytes": 4.0 * n * (1 + m) + sino, "flops": sweep}
    if op == "gradient":
        return {"bytes": 12.0 * n + sino, "flops": 2 * sweep}
    if op == "autograd":
        return {"bytes": 16.0 * n + sino, "flops": 3 * sweep}
    if op == "osem":
        return {"bytes": 4.0 * n * (1 + m) + sino, "flops": 2 * sweep * case["iterations"]}
    if op == "joint":  # twice: sensitivities, OSEM pass, projection and mu gradient
        return {"bytes": 16.0 * n + sino, "flops": 2 * 5 * sweep}
    return {"bytes": 4.0 * n * (2 + m) + sino, "flops": 3 * sweep}  # mlem_step


# ---- the same operations in double precision ------------------------------------

class _Exact:
    """The projector and its relatives in plain torch on (z, x, y)-ordered volumes."""

    def __init__(self, n, ny, cams, psf, dtype, dev):
        self.n, self.ny, self.dt, self.dev = n, ny, dtype, dev
        cams = np.asarray(cams, np.float64)
        self.ang = cams if cams.ndim == 2 else np.stack([0 * cams, cams, 0 * cams])
        self.V = self.ang.shape[1]
        self.tilt = bool(np.any(self.ang[0]) or np.any(self.ang[2]))
        self.Ty = self.Tx = None
        if psf is not None:
            p = psf.astype(np.float64)
            c = (p.shape[1] - 1) // 2
            self.Tx = self._banded(p[:, c, :], n)
            self.Ty = self._banded(p[:, :, c] / p[:, c, c][:, None], ny)

    def _banded(self, k, size):
        """(planes, size, size) matrices T with out = T in, the convolution
        out[i] = sum_j in[i + j] k[c - j] with zeros beyond the ends."""
        c = (k.shape[1] - 1) // 2
        i = torch.arange(size, device=self.dev)
        d = c - (i.view(1, -1) - i.view(-1, 1))
        kk = torch.from_numpy(k).to(self.dev, self.dt)
        return kk[:, d.clamp(0, 2 * c)] * ((d >= 0) & (d <= 2 * c))

    def blur(self, u, transpose=False):
        """The PSF of every plane of u (z, x, y), or its transpose."""
        if self.Tx is None:
            return u
        tx = self.Tx.transpose(1, 2).contiguous() if transpose else self.Tx
        ty = self.Ty if transpose else self.Ty.transpose(1, 2).contiguous()
        return torch.bmm(torch.bmm(tx, u.contiguous()), ty)

    def matrix(self, v):
        ax, ay, az = (float(a) for a in self.ang[:, v])
        rx = np.array([[1, 0, 0], [0, np.cos(ax), -np.sin(ax)], [0, np.sin(ax), np.cos(ax)]])
        ry = np.array([[np.cos(ay), 0, np.sin(ay)], [0, 1, 0], [-np.sin(ay), 0, np.cos(ay)]])
        rz = np.array([[np.cos(az), -np.sin(az), 0], [np.sin(az), np.cos(az), 0], [0, 0, 1]])
        return rz @ ry @ rx

    def corners(self, R):
        """[(flat index, weight, row?)] of the sample positions R (v - c) + c."""
        n, ny, dt, dev = self.n, self.ny, self.dt, self.dev
        c, cy = (n - 1) / 2.0, (ny - 1) / 2.0
        g = torch.arange(n, device=dev, dtype=dt)
        z, x = g.view(-1, 1, 1) - c, g.view(1, -1, 1) - c
        y = (torch.arange(ny, device=dev, dtype=dt) - cy).view(1, 1, -1) if self.tilt else None
        px, pz = R[0, 0] * x + R[0, 2] * z, R[2, 0] * x + R[2, 2] * z
        if self.tilt:
            px, pz = px + R[0, 1] * y, pz + R[2, 1] * y
            py = R[1, 0] * x + R[1, 1] * y + R[1, 2] * z + cy
        px, pz = px + c, pz + c

        def axis(p, size):
            f = torch.floor(p)
            out = []
            for q, w in ((f, 1 - (p - f)), (f + 1, p - f)):
                ok = (q >= 0) & (q < size)
                out.append((q.clamp(0, size - 1).long(), w * ok))
            return out

        res = []
        for iz, wz in axis(pz, n):
            for ix, wx in axis(px, n):
                if not self.tilt:
                    res.append(((iz * n + ix).reshape(-1), (wz * wx).reshape(-1, 1)))
                else:
                    for iy, wy in axis(py, ny):
                        res.append((((iz * n + ix) * ny + iy).reshape(-1), (wz * wx * wy).reshape(-1)))
        return res

    def pull(self, vol, cor):
        src = vol.reshape(-1) if self.tilt else vol.reshape(self.n * self.n, self.ny)
        out = None
        for i, w in cor:
            t = src.index_select(0, i) * w
            out = t if out is None else out + t
        return out.view(self.n, self.n, self.ny)

    def push(self, vol, cor, out):
        """out += the transpose of pull."""
        dst = out.view(-1) if self.tilt else out.view(self.n * self.n, self.ny)
        src = vol.reshape(-1) if self.tilt else vol.reshape(self.n * self.n, self.ny)
        for i, w in cor:
            dst.index_add_(0, i, src * w)

    def zxy(self, t):  # (z, y, x) -> (z, x, y)
        return None if t is None else t.to(self.dev, self.dt).permute(0, 2, 1).contiguous()

    def factors(self, mu, cor):
        return None if mu is None else torch.exp(-torch.cumsum(self.pull(mu, cor), 0))

    def project(self, act, mu, views=None):
        a, m = self.zxy(act), self.zxy(mu)
        out = []
        for v in range(self.V) if views is None else views:
            cor = self.corners(self.matrix(v))
            h, e = self.blur(self.pull(a, cor)), self.factors(m, cor)
            out.append((h if e is None else h * e).sum(0).t())
        return torch.stack(out)

    def backproject(self, sino, mu, views=None, adjoint=False):
        m = self.zxy(mu)
        acc = torch.zeros((self.n, self.n, self.ny), device=self.dev, dtype=self.dt)
        for k, v in enumerate(range(self.V) if views is None else views):
            R = self.matrix(v)
            cor = self.corners(R)
            s = sino[k].to(self.dev, self.dt).t().unsqueeze(0)
            e = self.factors(m, cor)
            u = s * e if e is not None else s.expand(self.n, -1, -1)
            u = self.blur(u, transpose=adjoint)
            if adjoint:
                self.push(u, cor, acc)
            else:
                acc += self.pull(u.contiguous(), self.corners(R.T))
        return acc.permute(0, 2, 1).contiguous()

    def gradient(self, sino, act, mu, exact):
        """The gradient in mu of <sino, project(act, mu)> (exact), or the
        reference's (PSF after the sum, inverse-rotation pull)."""
        a, m = self.zxy(act), self.zxy(mu)
        acc = torch.zeros((self.n, self.n, self.ny), device=self.dev, dtype=self.dt)
        for v in range(self.V):
            R = self.matrix(v)
            cor = self.corners(R)
            h = self.pull(a, cor)
            h = (self.blur(h) if exact else h) * self.factors(m, cor)
            tail = torch.flip(torch.cumsum(torch.flip(h, [0]), 0), [0])
            u = sino[v].to(self.dev, self.dt).t().unsqueeze(0) * tail
            if exact:
                self.push(-u, cor, acc)
            else:
                acc += self.pull(self.blur(u), self.corners(R.T))
        return acc.permute(0, 2, 1).contiguous()

    def em(self, x, counts, mu, subsets, iterations):
        order = [list(range(s, self.V, subsets)) for s in range(subsets)]
        sens = [self.backproject(torch.ones((len(o), self.ny, self.n)), mu, o).clamp_min(EPS) for o in order]
        for _ in range(iterations):
            for s, o in enumerate(order):
                p = self.project(x, mu, o).clamp_min(0)
                y = counts[o].to(self.dev, self.dt)
                b = self.backproject(torch.where(p < EPS, y / EPS, y / p), mu, o).clamp_min(0)
                x = x * (b / sens[s])
        return x


def exact(case, seed):
    dev = torch.device("cuda:0")
    f64 = torch.float64
    op = case["op"]
    if op == "batch":
        res = []
        for i in range(case["problems"]):
            p = _batch_problem(case["pick"], i)
            w = _problem(p, 100 * seed + i, dev)
            g = _Exact(p["n"], p["ny"], w["cameras"], w["psf"], f64, dev)
            res.append(g.em(torch.ones_like(w["activity"], dtype=f64), w["counts"], w["mu"], case["subsets"],
                            case["iterations"]))
        return res
    w = _problem(case, seed, dev)
    act, mu = w["activity"], w["mu"]
    g = _Exact(case["n"], case["ny"], w["cameras"], w["psf"], f64, dev)
    one = torch.ones_like(act, dtype=f64)
    if op == "project":
        return g.project(act, mu).clamp_min(0)
    if op == "backproject":
        return g.backproject(w["weights"], mu, adjoint=case["adjoint"]).clamp_min(0)
    if op == "gradient":
        return g.gradient(w["weights"], act, mu, False).clamp_min(0)
    if op == "autograd":
        act, mu, y = act * 0.9 + 0.05, mu * 0.8, w["counts"].to(f64)
        p = g.project(act, mu)
        q = p.clamp_min(1e-8)
        loss = (p - y * torch.log(q)).sum()
        weight = 1 - torch.where(p >= 1e-8, y / q, torch.zeros_like(p))
        return loss, g.backproject(weight, mu, adjoint=True), g.gradient(weight, act, mu, True)
    if op == "osem":
        return g.em(one, w["counts"], mu, case["subsets"], case["iterations"])
    if op == "joint":
        x, mu, y = one, (mu * 0.8).to(f64), w["counts"].to(f64)
        for _ in range(2):
            x = g.em(x, y, mu, case["subsets"], 1)
            p = g.project(x, mu)
            q = p.clamp_min(1e-8)
            grad = g.gradient(1 - torch.where(p >= 1e-8, y / q, torch.zeros_like(p)), x, mu, True)
            mu = (mu - 0.01 * grad / grad.abs().max().clamp_min(1e-30)).clamp_min(0)
        return x, mu, grad
    if op == "mlem_step":
        return g.em(one, w["counts"], mu, 1, 1)
    raise ValueError(op)
