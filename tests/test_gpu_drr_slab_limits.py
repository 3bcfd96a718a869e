"""Slab boxes where coordinates are large in voxels: a source far from the volume, a volume far from the
world's origin, and an axis of several 10^5 voxels. The march's values are those of rays shared by waves,
which gather, bit for bit; a box too narrow by its bounds' rounding would miss voxels at its edges."""
import numpy as np
import pytest

from tests.helpers import poses_f32

pytestmark = pytest.mark.gpu


def _both(monkeypatch, ctx, X, vol, cam, poses, step, **kw):
    out = []
    for reuse in ("1", "0"):
        monkeypatch.setenv("XRH_CELL_REUSE", reuse)
        n, px = len(poses), cam.num_det_rows * cam.num_det_cols
        buf = ctx.alloc(4 * n * px)
        X.line_int(ctx, vol, [cam], poses_f32(poses), np.zeros(n, np.int64), step, buf, **kw)
        out.append(buf.download(np.float32))
        buf.free()
    return out


@pytest.mark.parametrize("geom", [0, 1])
@pytest.mark.parametrize("focal,offset", [(3.0e4, 0.0), (2.0e5, 0.0), (3.0e5, 0.0), (2.0e3, 1.0e5)])
def test_far_source_and_far_origin(ctx, focal, offset, geom, monkeypatch):
    from xreg_amd import _xrh as X
    from xreg_amd import geometry as G
    from xreg_amd import synth

    print(f"case: slab limits, source {focal} away, origin {offset}, geom {geom}", flush=True)
    rng = np.random.default_rng(1)
    vox = rng.uniform(0.01, 0.05, (60, 1000, 56)).astype(np.float32)  # z, y, x: long along the rays
    i2p = np.array(G.idx_to_phys(1.0), np.float32).copy().reshape(4, 4)
    i2p[:3, 3] = offset
    vol = X.Volume(ctx, vox, i2p)
    center = np.array([28.0, 500.0, 30.0]) + offset
    # the detector 600 voxels behind the centre, about one voxel between rays
    cam = G.camera(focal, 50, 45, focal / (focal - 600.0), focal / (focal - 600.0))
    gt = G.gt_pose(center, focal - 600.0)
    poses = np.concatenate([gt[None], synth.random_poses(gt, center, 5, 2.0, 3.0, seed=4)])
    a, b = _both(monkeypatch, ctx, X, vol, cam, poses, 0.7, geom=geom)
    assert a.max() > 0.0
    assert np.array_equal(a, b)
    vol.close()


@pytest.mark.parametrize("geom", [0, 1])
def test_long_axis(ctx, geom, monkeypatch):
    from xreg_amd import _xrh as X
    from xreg_amd import geometry as G

    print(f"case: slab limits, an axis of 400000 voxels, geom {geom}", flush=True)
    rng = np.random.default_rng(2)
    n = 400000
    vox = np.tile(rng.uniform(0.01, 0.05, (5, 1000, 6)).astype(np.float32), (1, n // 1000, 1))
    vol = X.Volume(ctx, vox, G.idx_to_phys(1.0))
    center = np.array([3.0, n / 2.0, 2.5])
    focal = 1.5 * n
    cam = G.camera(focal, 16, 16, 1.0, 1.0)
    a, b = _both(monkeypatch, ctx, X, vol, cam, G.gt_pose(center, 0.7 * n)[None], 1.3, geom=geom)
    assert a.max() > 0.0
    assert np.array_equal(a, b)
    vol.close()
