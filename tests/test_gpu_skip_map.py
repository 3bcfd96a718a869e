"""The empty-space map built on the device: DRRs with it equal DRRs without it bit for bit on volumes
of a few isolated voxels (a distance too large anywhere would skip one), at every brick size, on odd
and one-voxel-wide volumes, and it removes most samples."""
import numpy as np
import pytest

from tests.helpers import poses_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", ["1", "2", "3", "4"])
@pytest.mark.parametrize("shape", [(50, 61, 47), (33, 16, 130), (40, 40, 1), (1, 40, 40), (3, 2, 5)])  # z, y, x
def test_isolated_voxels(ctx, shape, shift, monkeypatch):
    from xreg_amd import _xrh as X
    from xreg_amd import geometry as G
    from xreg_amd import synth

    print(f"case: skip map {shape} shift {shift}", flush=True)
    rng = np.random.default_rng(sum(shape) + int(shift))
    vox = np.zeros(shape, np.float32)
    corners = [(0, 0, 0), tuple(s - 1 for s in shape)]
    for idx in corners + [tuple(int(rng.integers(0, s)) for s in shape) for _ in range(4)]:
        vox[idx] = rng.uniform(0.02, 0.05)
    sp = 2.0
    center = G.vol_center_phys(shape[::-1], sp)
    gt = G.gt_pose(center, 510.0)
    cam = G.camera(1020.0, 48, 40, 6.0, 6.0)
    poses = np.concatenate([gt[None], synth.random_poses(gt, center, 6, 180.0, 4.0, seed=3)])
    n = len(poses)
    out, counts = [], []
    for skip in ("1", "0"):
        monkeypatch.setenv("XRH_SKIP_BRICK_SHIFT", shift)
        monkeypatch.setenv("XRH_SKIP_EMPTY", skip)
        vol = X.Volume(ctx, vox, G.idx_to_phys(sp))
        buf = ctx.alloc(4 * n * 48 * 40)
        X.line_int(ctx, vol, [cam], poses_f32(poses), np.zeros(n, np.int64), 0.7, buf)
        out.append(buf.download(np.float32))
        counts.append(X.line_int_sample_count(ctx, vol, [cam], poses_f32(poses), np.zeros(n, np.int64), 0.7,
                                              evaluated=True))
        buf.free()
        vol.close()
    if min(shape) > 1:  # (a volume one voxel wide has no inside for a ray to cross)
        assert out[0].max() > 0.0
    assert np.array_equal(out[0], out[1])
    assert counts[0][0] == counts[1][0] == counts[1][1]
    assert counts[0][1] <= counts[0][0]
    if min(shape) >= 16:
        assert counts[0][1] < 0.9 * counts[0][0]
