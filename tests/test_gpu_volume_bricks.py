"""Bricks, settled orbits and the re-evaluation list of the volume kernels.

A voxel's bits depend on its coordinates alone: not on the brick or list it
is evaluated in, nor on whether its wave settled (and stopped iterating) or
not. Points in shuffled order share their waves with unrelated points, which
hardly ever settle together, so they are the general path to compare with.
"""
from __future__ import annotations

import numpy as np
import pytest

import lyapunov3d_amd as lyap
from tests.gpu_util import empty, to_numpy, torch_cuda

pytestmark = pytest.mark.gpu

PRECS = [lyap.PREC_PLAIN, lyap.PREC_PRODUCT, lyap.PREC_FP64]


@pytest.fixture(scope="module")
def ctx():
    torch_cuda()
    c = lyap.Context(0)
    yield c
    c.close()


def grid_points(lo, hi, n):
    """The volume's coordinates (x fastest) in float, as the kernels form them."""
    ax = [np.float32(a) + ((np.float32(b) - np.float32(a)) * np.arange(k, dtype=np.float32)) / np.float32(k)
          for a, b, k in zip(lo, hi, n)]
    z, y, x = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    return np.stack([x, y, z], axis=-1).reshape(-1, 3).astype(np.float32)


def shuffled(ctx, xyz, prm, seq, mode):
    torch = torch_cuda()
    order = np.random.default_rng(3).permutation(len(xyz))
    dev = torch.from_numpy(xyz[order]).cuda()
    out = empty(4 * len(xyz))
    torch.cuda.synchronize()
    ctx.calc_points(out.data_ptr(), dev.data_ptr(), len(xyz), prm, seq, mode)
    ctx.sync()
    got = np.empty(len(xyz), np.float32)
    got[order] = to_numpy(out, np.float32)[:len(xyz)]
    return got


def volume(ctx, lo, hi, n, prm, seq, mode, noalloc=False):
    count = n[0] * n[1] * n[2]
    out = empty(4 * count)
    (ctx.calc_volume_noalloc if noalloc else ctx.calc_volume)(out.data_ptr(), prm, seq, lo, hi, n, mode)
    ctx.sync()
    return to_numpy(out, np.float32)[:count]


# one voxel, ragged edges, thin grids (memory order), whole bricks; windows
# shorter than a block and than a period; periods around the block lengths
@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("n,seq,settle,accum", [
    ((1, 1, 1), "ABBAC", 100, 400), ((64, 64, 8), "ABBAC", 100, 400), ((67, 5, 9), "AB", 37, 203),
    ((130, 1, 1), "ABC", 100, 333), ((33, 31, 2), "A", 50, 500), ((20, 20, 20), "ABCABCCA", 200, 1000),
    ((16, 16, 16), "AABCBBACCABC", 7, 5), ((12, 12, 12), "ABC", 0, 1), ((17, 16, 15), "ABCABBCACABCCBAABCAB", 90, 700),
    ((16, 16, 16), "ABCABBCACABCCBAABCABC", 90, 700), ((16, 16, 16), "ABCABBCACABCCBAABCABCABCABBCAABC", 90, 700)])
def test_volume_equals_shuffled_points(ctx, n, seq, settle, accum, prec):
    prm = lyap.make_params(settle=settle, accum=accum)
    for lo, hi in (((2.0, 2.0, 2.0), (4.0, 4.0, 4.0)), ((0.0, 0.0, 0.0), (4.0, 4.0, 4.0)),
                   ((3.5, 3.5, 3.5), (4.2, 4.2, 4.2))):
        m = lyap.volume_mode(prec)
        a = volume(ctx, lo, hi, n, prm, seq, m)
        b = shuffled(ctx, grid_points(lo, hi, n), prm, seq, m)
        assert a.tobytes() == b.tobytes(), (lo, hi)


@pytest.mark.parametrize("n", [(1, 1, 1), (7, 3, 5), (40, 40, 12), (65, 64, 1)])
def test_every_listed_voxel_is_reevaluated(ctx, n):
    """A rule that lists every voxel: single parts overflow into the next ones."""
    prm = lyap.make_params(settle=100, accum=300)
    lo, hi = (2.0, 2.0, 2.0), (4.0, 4.0, 4.0)
    every = lyap.volume_mode(lyap.PREC_PRODUCT, fp64_margin=1e9)
    ref = volume(ctx, lo, hi, n, prm, "ABBAC", lyap.volume_mode(lyap.PREC_FP64))
    assert ctx.last_reevaluated() == 0
    for noalloc in (True, False):
        assert volume(ctx, lo, hi, n, prm, "ABBAC", every, noalloc).tobytes() == ref.tobytes(), noalloc
    assert ctx.last_reevaluated() == n[0] * n[1] * n[2]


def test_list_holds_what_the_rule_selects(ctx):
    n, prm, seq = (48, 40, 36), lyap.make_params(settle=100, accum=600), "ABCABCCA"
    lo, hi = (2.5, 2.5, 2.5), (4.0, 4.0, 4.0)
    torch = torch_cuda()
    xyz = grid_points(lo, hi, n)
    dev = torch.from_numpy(xyz).cuda()
    lam, h1, h2 = (empty(4 * len(xyz)) for _ in range(3))
    torch.cuda.synchronize()
    ctx.calc_points_halves(lam.data_ptr(), h1.data_ptr(), h2.data_ptr(), dev.data_ptr(), len(xyz), prm, seq)
    ctx.sync()
    lam, h1, h2 = (to_numpy(t, np.float32)[:len(xyz)] for t in (lam, h1, h2))
    with np.errstate(invalid="ignore"):
        want = ~(np.abs(lam) >= np.float32(0.01))
        want |= (np.where(h1 < h2, h1, h2) < np.float32(0.2)) & (np.abs(h1 - h2) > np.float32(1e-4))
    mode = lyap.volume_mode(lyap.PREC_PRODUCT, fp64_margin=0.01, converge_tau=1e-4, converge_band=0.2)
    got = volume(ctx, lo, hi, n, prm, seq, mode)
    assert ctx.last_reevaluated() == int(want.sum()) > 0
    f64 = volume(ctx, lo, hi, n, prm, seq, lyap.volume_mode(lyap.PREC_FP64))
    assert got.tobytes() == np.where(want, f64, lam).astype(np.float32).tobytes()
