"""Jittered frames refined by the reversing walk, one lane per ray.

A ray's arithmetic does not depend on the launch it runs in, so the bytes
equal those of the reference's launch shape and of the persistent levels.
"""
from __future__ import annotations

import numpy as np
import pytest

import lyapunov3d_amd as lyap
from tests.gpu_util import RenderBuffers, device_lights, torch_cuda

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    torch_cuda()
    c = lyap.Context(0)
    yield c
    c.close()


def scene(w, h, shift=0.0):
    prm, cam, lights, n = lyap.params_init()
    prm.settle, prm.accum, prm.depth = 18, 60, 64.0
    cam.C.x += shift
    lyap.cam_recalculate(cam, w, h, 1)
    lyap.lights_recalculate(lights, n)
    return prm, cam, lights, n


# one ray, one whole block, ragged edges, a period past the 16-slot window
@pytest.mark.parametrize("prec", [lyap.PREC_PLAIN, lyap.PREC_PRODUCT, lyap.PREC_FP64])
@pytest.mark.parametrize("w,h,seq", [(1, 1, "BCABA"), (8, 8, "BCABA"), (63, 5, "A"), (70, 33, "BCABA"),
                                     (33, 17, "ABCABBCACABCCBAABCA")])
def test_bytes_equal_the_other_schedules(ctx, w, h, seq, prec):
    prm, cam, lights, n = scene(w, h)
    ld = device_lights(lights, n)
    got = {}
    for sched in (lyap.SCHEDULE_BATCHED, lyap.SCHEDULE_LEVELS, lyap.SCHEDULE_DIRECT):
        b = RenderBuffers(w, h)
        b.render(ctx, cam, prm, seq, ld, n, lyap.render_mode(precision=prec, schedule=sched))
        ctx.sync()
        got[sched] = dict(b.fetch(), total=np.array(ctx.last_evals()))
    for sched in (lyap.SCHEDULE_LEVELS, lyap.SCHEDULE_DIRECT):
        for k, a in got[lyap.SCHEDULE_BATCHED].items():
            assert a.tobytes() == got[sched][k].tobytes(), (sched, k)


def test_batch_of_jittered_views(ctx):
    """Views of different sizes share the launch; each gets the bytes of a call of its own."""
    mode = lyap.render_mode(precision=lyap.PREC_PLAIN)
    views, bufs, alone = [], [], []
    for i, (w, h) in enumerate([(40, 24), (9, 50), (64, 64)]):
        prm, cam, lights, n = scene(w, h, 0.03 * i)
        prm.accum = 40 + 17 * i
        ld = device_lights(lights, n)
        one, b = RenderBuffers(w, h), RenderBuffers(w, h)
        one.render(ctx, cam, prm, "BCABA", ld, n, mode)
        ctx.sync()
        alone.append(one.fetch())
        bufs.append((b, ld))
        views.append(lyap.make_view(cam, prm, "BCABA", w, h, b.rgba.data_ptr(), b.points.data_ptr(),
                                    b.depth.data_ptr(), b.lam.data_ptr(), b.evals.data_ptr(), ld.data_ptr(), n))
    ctx.render_batch(views, mode)
    ctx.sync()
    for (b, _), ref in zip(bufs, alone):
        for k, a in b.fetch().items():
            assert a.tobytes() == ref[k].tobytes(), k
