"""Frames refined by bisection in march passes.

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


def scene(w, h, depth=64.0, shift=0.0, **fields):
    prm, cam, lights, n = lyap.params_init()
    prm.settle, prm.accum, prm.depth, prm.jitter = 18, 40, depth, 0.0
    for k, x in fields.items():
        setattr(prm, k, x)
    cam.C.x += shift
    lyap.cam_recalculate(cam, w, h, 1)
    lyap.lights_recalculate(lights, n)
    return prm, cam, lights, n


def mode(sched=lyap.SCHEDULE_BATCHED, prec=lyap.PREC_PRODUCT):
    return lyap.render_mode(precision=prec, refine=lyap.REFINE_BISECT, schedule=sched)


def frame(ctx, w, h, seq, prec, sched, **fields):
    prm, cam, lights, n = scene(w, h, **fields)
    ld = device_lights(lights, n)
    b = RenderBuffers(w, h)
    b.render(ctx, cam, prm, seq, ld, n, mode(sched, prec))
    ctx.sync()
    return dict(b.fetch(), total=np.array(ctx.last_evals()))


# one ray, ragged edges; each kind of step between passes (near and far
# steps, steps by the length in the box, jitter); marches of many samples, also
# past the length whose index and offset share a record's word; the two sides
# of the launch sizes that change the passes (200,000 rays) and the refining
# lanes as well (1.8 million), with ragged rows
@pytest.mark.parametrize("prec", [lyap.PREC_PLAIN, lyap.PREC_PRODUCT, lyap.PREC_FP64])
@pytest.mark.parametrize("w,h,fields", [
    (1, 1, {}), (70, 33, {}), (63, 5, {"nearMultiplier": 3.0}), (40, 41, {"stepMethod": 1, "nearMultiplier": 2.0}),
    (40, 41, {"stepMethod": 0}), (24, 17, {"jitter": 0.5}), (24, 17, {"jitter": 0.5, "stepMethod": 1}),
    (64, 64, {"depth": 2000.0}), (4, 3, {"depth": 80000.0, "stepMethod": 1}), (4, 3, {"depth": 80000.0, "stepMethod": 0}),
    (440, 440, {"depth": 48.0}), (449, 448, {"depth": 48.0}), (1344, 1336, {"depth": 16.0}), (1345, 1344, {"depth": 16.0, "nearMultiplier": 2.0})])
def test_bytes_equal_the_other_schedules(ctx, w, h, fields, prec):
    got = frame(ctx, w, h, "BCABA", prec, lyap.SCHEDULE_BATCHED, **fields)
    for sched in (lyap.SCHEDULE_LEVELS, lyap.SCHEDULE_DIRECT):
        ref = frame(ctx, w, h, "BCABA", prec, sched, **fields)
        for k, a in got.items():
            assert a.tobytes() == ref[k].tobytes(), (sched, k)


# 8 views: eight sub-lists each; 9: seven; 33 and 64: one; 65: the levels
@pytest.mark.parametrize("count", [8, 9, 33, 64, 65])
def test_batches(ctx, count):
    """Views of different sizes share the passes; each gets the bytes of a call of its own."""
    views, bufs, alone = [], [], []
    for i in range(count):
        w, h = 8 + 5 * (i % 7), 6 + 9 * (i % 5)
        prm, cam, lights, n = scene(w, h, shift=0.01 * (i % 11))
        ld = device_lights(lights, n)
        one, b = RenderBuffers(w, h), RenderBuffers(w, h)
        one.render(ctx, cam, prm, "BCABA", ld, n, mode(lyap.SCHEDULE_DIRECT))
        ctx.sync()
        alone.append(one.fetch())
        bufs.append((b, ld))
        views.append(lyap.make_view(cam, prm, "BCABA", w, h, b.rgba.data_ptr(), b.points.data_ptr(),
                                    b.depth.data_ptr(), b.lam.data_ptr(), b.evals.data_ptr(), ld.data_ptr(), n))
    ctx.render_batch(views, mode())
    ctx.sync()
    for (b, _), ref in zip(bufs, alone):
        for k, a in b.fetch().items():
            assert a.tobytes() == ref[k].tobytes(), k
