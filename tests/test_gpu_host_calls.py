"""Calls on host arrays share device blocks from one call to the next: whatever
an earlier call left in them (NaN here), and whatever other threads run at the
time, a call's result is the bits it has on fresh memory.  Shapes at the edges
of the paths: one voxel, the general path, sweeps, row-lane kernels, tiles."""
import threading

import numpy as np
import pytest

from niftyrec_amd import phantoms

pytestmark = pytest.mark.gpu

SHAPES = [((1, 1, 1), 0, False), ((24, 20, 24), 5, True), ((33, 31, 33), 5, False), ((40, 140, 40), 3, False),
          ((96, 40, 96), 7, False), ((80, 132, 80), 3, False)]


def _ops(shape, K, tilt, fill=None):
    from niftyrec_amd import api
    rng = np.random.default_rng(7)
    V = 6
    act, mu = rng.random(shape, dtype=np.float32), 0.02 * rng.random(shape, dtype=np.float32)
    sino = rng.random((V,) + shape[1:], dtype=np.float32)
    if fill is not None:
        act, mu, sino = (np.full_like(a, fill) for a in (act, mu, sino))
    cams = np.linspace(0.1, 5.0, V).astype(np.float32)
    if tilt:
        cams = np.stack([cams, 0.3 * cams, 0.1 * cams]).astype(np.float32)
    psf = phantoms.gaussian_psf(shape[2], K, 0.5, 1.6) if K else None
    ops = [lambda: api.project(act, cams, psf, mu), lambda: api.project(act, cams, psf),
           lambda: api.backproject(sino, cams, psf, mu), lambda: api.backproject(sino, cams, psf),
           lambda: api.gradient_attenuation(sino, act, mu, cams, psf),
           lambda: api.mlem_step(act, sino, cams, psf, mu), lambda: api.mlem_step(act, sino, cams, psf),
           lambda: api.rotate(act, (0.1, 0.2, 0.3), [(n - 1) / 2 for n in shape[::-1]])]
    if K:
        ops.append(lambda: api.convolve(act, psf))
    return ops


def _reset():
    from niftyrec_amd import _lib
    assert _lib.load().et_array_reset_gpu() == 0


@pytest.mark.parametrize("shape, K, tilt", SHAPES)
def test_blocks_left_by_other_calls(shape, K, tilt):
    ref = []
    for op in _ops(shape, K, tilt):
        _reset()
        ref.append(op())
    poison = _ops(shape, K, tilt, np.nan)
    for k, op in enumerate(_ops(shape, K, tilt)):
        for p in (poison[k], poison[5], poison[(k + 1) % len(poison)]):
            p()
        got = op()
        assert np.isfinite(got).all() and np.array_equal(got, ref[k]), k


def test_threads_share_the_blocks():
    ops = [op for s in SHAPES[:5] for op in _ops(*s)]
    ref = [op() for op in ops]
    bad = []

    def work(t):
        for i in range(2 * len(ops)):
            k = (i * 7 + 11 * t) % len(ops)
            if not np.array_equal(ops[k](), ref[k]):
                bad.append((t, k))

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    _reset()
    assert np.array_equal(ops[0](), ref[0])
