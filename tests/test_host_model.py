"""The host layer (et_host.cpp) on a CPU model of the device
(host_model/model.cpp): every launch's arguments are checked against the live
device blocks, and results carry tags of what they were formed from, so that a
call that used something stale differs from the same call on a fresh plan.
Failed allocations and launches are forced from here."""
import ctypes
import os
import subprocess

import pytest

from conftest import ROOT

P, I, F = ctypes.c_void_p, ctypes.c_int, ctypes.c_float
STREAM = P(0x700)
NO_LIMIT = (1 << 64) - 1
ALLOC_FAILED = 4  # niftyrec_error_allocgpu


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("model") / "libmodel.so")
    csrc = os.path.join(ROOT, "niftyrec_amd", "csrc")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-w", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                           "-D__align__(x)=__attribute__((aligned(x)))", "-DHIP_SYMBOL(x)=x", "-I/opt/rocm/include",
                           "-I" + os.path.join(ROOT, "include"), "-I" + csrc, os.path.join(csrc, "et_host.cpp"),
                           os.path.join(ROOT, "tests", "host_model", "model.cpp"), "-Wl,-Bsymbolic", "-Wl,-z,defs",
                           "-o", out])
    m = ctypes.CDLL(out)
    for name, res, args in (("model_volume", P, [ctypes.c_size_t, ctypes.c_ulonglong]),
                            ("model_set", None, [P, ctypes.c_ulonglong]), ("model_tag", ctypes.c_ulonglong, [P]),
                            ("model_violations", ctypes.c_char_p, []), ("model_used", ctypes.c_size_t, []),
                            ("model_limit", None, [ctypes.c_size_t]), ("model_fail", None, [ctypes.c_char_p, I]),
                            ("model_count", I, [ctypes.c_char_p]), ("model_begin", None, [P]),
                            ("model_replay", None, [I]),
                            ("et_plan_create", I, [P, I, I, I, P, I, I, P, I, F, F]), ("et_plan_destroy", I, [P]),
                            ("et_plan_project", I, [P, P, P, P, I, P]),
                            ("et_plan_backproject", I, [P, P, P, P, I, I, P]),
                            ("et_plan_gradient_attenuation", I, [P, P, P, P, P, I, I, P]),
                            ("et_plan_project_backward", I, [P, P, P, P, P, P, I, P]),
                            ("et_plan_osem", I, [P, P, P, P, I, I, F, P]), ("et_plan_set_mu_check", I, [P, I]),
                            ("et_plan_set_tuning", I, [P, I, I]), ("et_plan_invalidate", I, [P])):
        getattr(m, name).restype = res
        getattr(m, name).argtypes = args
    yield m
    assert m.model_violations() == b""


class Rig:
    """Plans of one geometry (nx, ny, nz, views) and the volumes they work on."""

    def __init__(self, model, nx, ny, nz, views, psf=0, cols=1, bg=0.0):
        self.m, self.dims, self.V, self.K, self.cols, self.bg = model, (nx, ny, nz), views, psf, cols, bg
        model.model_clear()
        model.model_limit(NO_LIMIT)
        self.seq = 100
        self.plans, self.vols = [], []

    def plan(self):
        nx, ny, nz = self.dims
        cams = (F * (self.V * self.cols))(*[0.1 + 0.3 * i for i in range(self.V * self.cols)])
        psf = None if not self.K else (F * (self.K * self.K * nz))(*([0.5] * (self.K * self.K * nz)))
        h = P()
        assert self.m.et_plan_create(ctypes.byref(h), nx, ny, nz, cams, self.V, self.cols, psf, self.K, self.bg,
                                     0.0) == 0
        assert self.m.et_plan_set_mu_check(h, 0) == 0
        self.plans.append(h)
        return h

    def vol(self, sino=False):
        nx, ny, nz = self.dims
        self.seq += 1
        v = P(self.m.model_volume(nx * ny * (self.V if sino else nz), self.seq))
        self.vols.append(v)
        return v

    def tag(self, v):
        return self.m.model_tag(v)

    def project(self, h, a, m, out, truncate=1):
        return self.m.et_plan_project(h, a, m, out, truncate, STREAM)

    def backproject(self, h, s, m, out, adjoint=0, truncate=1):
        return self.m.et_plan_backproject(h, s, m, out, adjoint, truncate, STREAM)

    def gradient(self, h, s, a, m, out, exact=1, truncate=1):
        return self.m.et_plan_gradient_attenuation(h, s, a, m, out, exact, truncate, STREAM)

    def backward(self, h, s, a, m, ga, gm):
        return self.m.et_plan_project_backward(h, s, a, m, ga, gm, 0, STREAM)

    def osem(self, h, x, y, m, subsets, eps=1e-6, iterations=1):
        return self.m.et_plan_osem(h, x, y, m, subsets, iterations, eps, STREAM)

    def close(self):
        for h in self.plans:
            assert self.m.et_plan_destroy(h) == 0
        assert self.m.model_violations() == b""
        for v in self.vols:
            self.m.hipFree(v)


@pytest.mark.parametrize("op", ["gradient", "backward"])
@pytest.mark.parametrize("spare", [0, 30000, 250000, 500000])
def test_gradient_after_a_failed_allocation(model, op, spare):
    """A gradient that ran out of memory leaves no forward sums behind: the next
    one of the same activity and map forms them, whatever was projected before."""
    r = Rig(model, 40, 20, 32, 4)
    A, B, M, S, out, out2 = r.vol(), r.vol(), r.vol(), r.vol(sino=True), r.vol(), r.vol()

    def call(h, a):
        return r.gradient(h, S, a, M, out) if op == "gradient" else r.backward(h, S, a, M, out2, out)

    plan = r.plan()
    assert r.project(plan, A, M, S) == 0
    model.model_set(S, 7)
    model.model_limit(model.model_used() + spare)
    assert call(plan, B) in (0, ALLOC_FAILED)
    model.model_limit(NO_LIMIT)
    assert call(plan, B) == 0
    got = r.tag(out)
    assert call(r.plan(), B) == 0
    assert got == r.tag(out)
    r.close()


@pytest.mark.parametrize("op", ["gradient", "reference gradient", "backproject"])
@pytest.mark.parametrize("chunks", [0, 1])
def test_osem_after_an_operation_ran_out_of_memory(model, op, chunks):
    """Operations share their work buffers with OSEM.  Whatever an operation that
    found no room left of them, the next OSEM call has buffers of the size its
    launches use."""
    for spare in range(-1300000, 3000000, 100000):
        r = Rig(model, 40, 20, 32, 12)
        A, M, X, Y, S, out = r.vol(), r.vol(), r.vol(), r.vol(sino=True), r.vol(sino=True), r.vol()

        def osem(h):
            model.model_set(X, 5)
            assert r.osem(h, X, Y, M, 3) == 0
            return r.tag(X)

        plan, fresh = r.plan(), r.plan()
        for h in (plan, fresh):
            assert model.et_plan_set_tuning(h, chunks, 0) == 0
        ref = osem(fresh)
        assert osem(plan) == ref
        model.model_limit(max(0, model.model_used() + spare))
        if op == "backproject":
            r.backproject(plan, S, None, out, 1)
        else:
            r.gradient(plan, S, A, M, out, exact=int(op == "gradient"))
        model.model_limit(NO_LIMIT)
        assert osem(plan) == ref
        assert model.model_violations() == b""
        r.close()


def test_scarce_memory_keeps_the_views_that_fit(model):
    """Rotated-frame volumes for fewer views than asked for are kept from call to
    call: no buffer is freed and asked for again."""
    r = Rig(model, 40, 20, 32, 12)
    S, out = r.vol(sino=True), r.vol()
    big = r.plan()
    before = model.model_used()
    assert r.backproject(big, S, None, out) == 0
    whole = model.model_used() - before
    plan = r.plan()
    model.model_limit(model.model_used() + whole - 400000)  # not the volumes of all 12 views
    assert r.backproject(plan, S, None, out) == 0
    assert model.model_count(b"fill") > 0
    model.model_clear()
    for _ in range(3):
        assert r.backproject(plan, S, None, out) == 0
    assert model.model_count(b"fill") == 0
    r.close()


@pytest.mark.parametrize("failing", ["yl_sweep", "yl_pull", "planes_t"])
@pytest.mark.parametrize("nth", [1, 2, 3])
def test_epsilon_after_a_failed_osem_call(model, failing, nth):
    """An OSEM call with another epsilon that fails on its way leaves nothing of
    that epsilon to the next call."""
    r = Rig(model, 40, 20, 32, 6)
    M, X, Y = r.vol(), r.vol(), r.vol(sino=True)

    def osem(h, eps):
        model.model_set(X, 5)
        return r.osem(h, X, Y, M, 2, eps)

    plan, fresh = r.plan(), r.plan()
    assert osem(fresh, 0.5) == 0
    ref = r.tag(X)
    assert osem(plan, 0.5) == 0
    model.model_fail(failing.encode(), nth)
    osem(plan, 0.25)
    model.model_fail(b"", 0)
    assert osem(plan, 0.5) == 0
    assert r.tag(X) == ref
    r.close()


class Calls:
    """The single operations and OSEM on one plan's buffers, and on a fresh plan
    for comparison."""

    def __init__(self, r):
        self.r = r
        self.A, self.B, self.M, self.N = (r.vol() for _ in range(4))
        self.S, self.Y = r.vol(sino=True), r.vol(sino=True)

    def outputs(self):
        r = self.r
        return dict(sino=r.vol(sino=True), img=r.vol(), img2=r.vol())

    def call(self, h, op, o):
        r = self.r
        st = {"project A M": lambda: r.project(h, self.A, self.M, o["sino"]),
              "project B M": lambda: r.project(h, self.B, self.M, o["sino"]),
              "project A N": lambda: r.project(h, self.A, self.N, o["sino"]),
              "project A": lambda: r.project(h, self.A, None, o["sino"]),
              "adjoint": lambda: r.backproject(h, self.S, None, o["img"], 1, 0),
              "reference": lambda: r.backproject(h, self.S, None, o["img"], 0, 1),
              "adjoint M": lambda: r.backproject(h, self.S, self.M, o["img"], 1, 0),
              "gradient A M": lambda: r.gradient(h, self.S, self.A, self.M, o["img"]),
              "gradient B N": lambda: r.gradient(h, self.S, self.B, self.N, o["img"]),
              "reference gradient": lambda: r.gradient(h, self.S, self.A, self.M, o["img"], 0),
              "backward A M": lambda: r.backward(h, self.S, self.A, self.M, o["img"], o["img2"]),
              "osem M": lambda: r.osem(h, o["img"], self.Y, self.M, 2),
              "osem": lambda: r.osem(h, o["img"], self.Y, None, 2)}[op]
        if op.startswith("osem"):
            r.m.model_set(o["img"], 9)
        return st()

    def tags(self, o):
        return [self.r.tag(v) for v in o.values()]

    def fresh(self, op):
        o = self.outputs()
        for v in o.values():
            self.r.m.model_set(v, 3)
        assert self.call(self.r.plan(), op, o) == 0
        return self.tags(o)


CAPTURED = ["project A M", "project A", "adjoint", "adjoint M", "gradient A M", "reference gradient", "backward A M",
            "osem M", "osem"]
BETWEEN = ["project B M", "project A N", "project A", "adjoint", "reference", "gradient B N", "gradient A M",
           "rewrite", "invalidate", "osem M"]


@pytest.mark.parametrize("op", CAPTURED)
def test_captured_calls(model, op):
    """A captured call gives at every replay what the call gives on a fresh plan
    then, whatever ran in between; so do the calls after a replay."""
    r = Rig(model, 40, 20, 32, 6)
    c = Calls(r)
    plan, o, e = r.plan(), c.outputs(), c.outputs()
    for warm in BETWEEN + [op]:  # every buffer has its size, and the caches are some other map's
        if warm not in ("rewrite", "invalidate"):
            assert c.call(plan, warm, e) == 0
    if op.startswith("osem"):
        assert c.call(plan, op, o) == 0  # (the caches are built by a call of its own)
    model.model_begin(STREAM)
    assert c.call(plan, op, o) == 0
    g = model.model_end()

    def replay():
        for v in o.values():
            model.model_set(v, 9 if op.startswith("osem") else 3)
        model.model_replay(g)
        got = c.tags(o)
        ref = c.fresh(op)
        if op.startswith("osem"):
            got, ref = got[1:2], ref[1:2]
        assert got == ref

    replay()
    for step, between in enumerate(BETWEEN):
        if op.startswith("osem") and between in ("osem M", "rewrite", "invalidate"):
            continue  # (the caller's part: the sensitivities are the captured call's)
        if between == "rewrite":
            model.model_set(c.M, 1000 + step)
            model.model_set(c.A, 2000 + step)
        elif between == "invalidate":
            assert model.et_plan_invalidate(plan) == 0
        else:
            for v in e.values():
                model.model_set(v, 3)
            assert c.call(plan, between, e) == 0
            got, ref = c.tags(e), c.fresh(between)
            if between.startswith("osem"):
                got, ref = got[1:2], ref[1:2]
            assert got == ref, between
        replay()
        replay()
    r.close()


def test_a_captured_call_that_never_ran(model):
    """Capturing changes nothing that later calls rely on."""
    r = Rig(model, 40, 20, 32, 6)
    c = Calls(r)
    plan, e = r.plan(), c.outputs()
    for warm in BETWEEN + ["backward A M"]:
        if warm not in ("rewrite", "invalidate"):
            assert c.call(plan, warm, e) == 0
    for captured in CAPTURED[:-2]:
        for after in ["gradient A M", "gradient B N", "project A N", "adjoint M", "osem M"]:
            model.et_plan_invalidate(plan)
            model.model_begin(STREAM)
            assert c.call(plan, captured, e) == 0
            model.model_end()
            for v in e.values():
                model.model_set(v, 3)
            assert c.call(plan, after, e) == 0
            got, ref = c.tags(e), c.fresh(after)
            if after.startswith("osem"):
                got, ref = got[1:2], ref[1:2]
            assert got == ref, (captured, after)
    r.close()


def test_no_rebuild_is_captured(model):
    """An OSEM call that would build its caches is refused under capture, and the
    next call builds them."""
    r = Rig(model, 40, 20, 32, 6)
    c = Calls(r)
    plan, o = r.plan(), c.outputs()
    assert c.call(plan, "osem M", o) == 0
    model.et_plan_invalidate(plan)
    model.model_begin(STREAM)
    assert c.call(plan, "osem M", o) != 0
    model.model_end()
    assert c.call(plan, "osem M", o) == 0
    assert c.tags(o)[1] == c.fresh("osem M")[1]
    r.close()


def test_tables_are_bounded(model):
    """Calls of ever other kinds do not pile up tables."""
    r = Rig(model, 40, 20, 32, 6)
    c = Calls(r)
    plan, o = r.plan(), c.outputs()
    for i in range(60):
        if i == 30:
            held = model.model_used()
        for d in range(1, 7):
            assert model.et_plan_set_tuning(plan, 1 + i % 8, d) == 0
            assert c.call(plan, "adjoint", o) == 0
            assert c.call(plan, "project A", o) == 0
    assert model.model_used() == held
    r.close()


@pytest.mark.parametrize("dims, views, cols", [((72, 130, 8), 4, 1), ((200, 20, 8), 4, 1), ((40, 20, 32), 4, 1)])
@pytest.mark.parametrize("op", ["project A M", "project A", "adjoint", "adjoint M", "gradient A M",
                                "reference gradient", "backward A M"])
def test_more_memory_never_refuses_a_call(model, dims, views, cols, op):
    """An operation that the sweep kernels can do in the memory there is is done,
    also where the row-lane kernels' factors fit and their other buffers do not."""
    r = Rig(model, *dims, views, cols=cols)
    c = Calls(r)
    o = c.outputs()
    base = r.plan()
    before = model.model_used()
    assert c.call(base, op, o) == 0
    most = model.model_used() - before
    model.et_plan_destroy(r.plans.pop())
    ok = []
    for i in range(41):
        plan = r.plan()
        model.model_limit(model.model_used() + most * i // 40)
        ok.append(c.call(plan, op, o) == 0)
        model.model_limit(NO_LIMIT)
        assert c.call(plan, op, o) == 0
        model.et_plan_destroy(r.plans.pop())
    assert ok == sorted(ok), ok
    r.close()


@pytest.mark.parametrize("first", ["project A M", "backward A M", "adjoint"])
@pytest.mark.parametrize("op", ["osem M", "osem", "reference gradient", "adjoint M"])
def test_kept_buffers_give_way(model, first, op):
    """What a plan keeps of an operation (factors of every view, sums, planes) is
    given back where another of its calls finds no room."""
    r = Rig(model, 72, 130, 16, 8)
    c = Calls(r)
    o = c.outputs()
    probe = r.plan()
    before = model.model_used()
    for limit in range(0, 1 << 26, 1 << 17):  # what the call alone can do with
        model.model_limit(before + limit)
        if c.call(probe, op, o) == 0:
            break
    least = limit
    model.model_limit(NO_LIMIT)
    model.et_plan_destroy(r.plans.pop())
    plan = r.plan()
    before = model.model_used()
    assert c.call(plan, first, o) == 0
    model.model_limit(before + least + (3 << 20))  # (and the packed volumes, which any operation keeps)
    assert c.call(plan, op, o) == 0
    model.model_limit(NO_LIMIT)
    for again in (first, op):
        for v in o.values():
            model.model_set(v, 3)
        assert c.call(plan, again, o) == 0
        if not again.startswith("osem"):
            assert c.tags(o) == c.fresh(again)
    r.close()


@pytest.mark.parametrize("dims, views, chunks", [((1, 1, 1), 70000, 0), ((2, 1, 66000), 2, 0), ((1, 1, 8), 40000, 4)])
def test_general_path_beyond_a_grid(model, dims, views, chunks):
    """More views, planes, or views in chunks than a launch has blocks along an axis."""
    r = Rig(model, *dims, views, cols=3)
    A, S, out = r.vol(), r.vol(sino=True), r.vol()
    plan = r.plan()
    assert model.et_plan_set_tuning(plan, chunks, 0) == 0
    assert r.project(plan, A, A, S) == 0
    assert r.backproject(plan, S, None, out) == 0
    assert r.gradient(plan, S, A, A, out) == 0
    r.close()


@pytest.mark.parametrize("axis", [0, 1])
def test_random_subsets_wait_for_their_records(model, axis):
    """The random-subset driver builds its plan anew for every step: no record is
    overwritten that a launch of the step before may still read."""
    model.model_clear()
    model.model_limit(NO_LIMIT)
    n, ny, V = 8, 6, 12
    floats = lambda k: (F * k)(*([1.0] * k))  # noqa: E731
    x, y, mu, psf = floats(n * n * ny), floats(n * ny * V), floats(n * n * ny), floats(9 * n)
    f = model.et_array_osem
    f.argtypes = [P, ctypes.c_uint, ctypes.c_uint, ctypes.c_uint, P, I, F, F, ctypes.c_uint, I, I, P, I, P,
                  ctypes.c_uint, ctypes.c_uint, F, F, F, I]
    assert f(x, n, ny, 4, y, V, 0.0, 360.0, axis, 3, 1, mu, 1, psf, 3, 3, 0.0, 0.0, 1e-6, 1) == 0
    assert model.model_violations() == b""


@pytest.mark.parametrize("dims, views, planes", [((100, 192, 100), 40, 34), ((192, 200, 192), 12, 28),
                                                 ((65, 130, 65), 40, 22), ((256, 250, 256), 90, 396)])
def test_a_tall_projection_ends_in_full_rounds(model, dims, views, planes):
    """The depth chunks of a tall plan's projection without attenuation (one block
    per CU at a time): rounds of 256 blocks, times the planes of a block, are within
    a tenth of the planes of all blocks over 256."""
    r = Rig(model, *dims, views)
    assert r.project(r.plan(), r.vol(), None, r.vol(sino=True)) == 0
    assert -(-model.model_sweep_blocks() // 256) * model.model_sweep_planes() <= planes
    r.close()


@pytest.mark.parametrize("dims, psf, tiles", [((100, 130, 100), 21, (0, 0)), ((100, 130, 100), 3, (0, 1)),
                                              ((100, 130, 100), 0, (1, 1)), ((65, 192, 65), 11, (1, 1)),
                                              ((192, 192, 192), 7, (1, 1)), ((192, 200, 192), 21, (0, 0)),
                                              ((256, 40, 256), 21, (0, 0)), ((224, 64, 224), 21, (1, 1)),
                                              ((193, 17, 193), 11, (1, 1))])
def test_backprojections_take_the_faster_kernels(model, dims, psf, tiles):
    """Wide and tall plans without attenuation, (reference, adjoint): tile kernels
    or not, as timed."""
    r = Rig(model, *dims, 2, psf=psf)
    plan, S, out = r.plan(), r.vol(sino=True), r.vol()
    for adjoint in (0, 1):
        model.model_clear()
        assert r.backproject(plan, S, None, out, adjoint) == 0
        assert (model.model_count(b"yl_sweep") > 0) == bool(tiles[adjoint])
    r.close()
