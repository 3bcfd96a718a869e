"""Contexts with an HBM budget keep no plain voxels, so their rays gather: the same DRRs and similarities
as a context without a budget, over a volume large enough to be taken by slabs there, through casts, batches
(graph replays) and several objects, for FP32 and 16-bit storage."""
import numpy as np
import pytest

from tests.helpers import poses_f32

pytestmark = pytest.mark.gpu

SHAPE = (170, 161, 163)  # z, y, x: 72 MB of cells


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("spacing", [0.5, 0.8, 1.3, 3.0])
@pytest.mark.parametrize("geom", [0, 1])
def test_budget_equals_no_budget(ctx, storage, spacing, geom):
    from xreg_amd import _xrh as X
    from xreg_amd import geometry as G
    from xreg_amd import synth

    print(f"case: budget storage {storage} spacing {spacing} geom {geom}", flush=True)
    rng = np.random.default_rng(8)
    vox = (rng.uniform(0.01, 0.05, SHAPE) * (rng.uniform(size=SHAPE) < 0.8)).astype(np.float32)
    center = G.vol_center_phys(SHAPE[::-1], 1.0)
    gt = G.gt_pose(center, 510.0)
    rows, cols = 130, 117
    cam = G.camera(1020.0, rows, cols, 2.0 * spacing, 2.0 * spacing)
    # 72 tiles a pose: enough poses that whole rays are cast
    poses = np.concatenate([gt[None], synth.random_poses(gt, center, 35, 30.0, 5.0, seed=2)])
    n, npx = len(poses), rows * cols
    fixed = rng.random((rows, cols), dtype=np.float32)
    got = []
    for c in (ctx, X.Context(0, hbm_budget_bytes=4 << 30)):
        vol = X.Volume(c, vox, G.idx_to_phys(1.0), storage=storage)
        buf = c.alloc(4 * n * npx)
        X.line_int(c, vol, [cam], poses_f32(poses), np.zeros(n, np.int64), 0.6, buf, geom=geom)
        cast = buf.download(np.float32)
        fx = X.Fixed(c, fixed, X.XRH_SIM_NCC)
        b = X.Batch(c, [X.make_view(vol, fx, cam, 0.6)] * 2, max_items=n, geom=geom)
        sims = [b.eval(np.zeros(n, np.int32), poses, drr=buf) for _ in range(2)]
        assert np.array_equal(sims[0], sims[1])
        drr = buf.download(np.float32)
        pairs = poses.reshape(n // 2, 2, 4, 4)
        osims = [b.eval_objects(np.tile(np.arange(2, dtype=np.int32), (n // 2, 1)), pairs, drr=buf) for _ in range(2)]
        assert np.array_equal(osims[0], osims[1])
        both = buf.download(np.float32)[: n // 2 * npx]
        got.append((cast, sims[0], drr, osims[0], both))
        for o in (b, fx, vol):
            o.close()
        buf.free()
        if c is not ctx:
            c.close()
    assert got[0][0].max() > 0.0
    for a, b in zip(*got):
        assert np.array_equal(a, b)
