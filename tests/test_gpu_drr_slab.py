"""Slab marching (large FP32 launches) and rays shared by several waves (small ones): both sum the
same samples in the same order, so their DRRs are equal bit for bit, at every viewing direction and
ray spacing (from boxes of many layers to boxes that do not fit, which gather), on ragged detectors,
volumes with edges of one and two voxels, for SUM and MAX and both ray set-ups."""
import numpy as np
import pytest

from tests.helpers import DRR_REL_TOL, drr_rel_err, poses_f32

pytestmark = pytest.mark.gpu

SHAPES = {"box": (33, 20, 47), "odd": (65, 70, 63), "flat_x": (40, 44, 1), "flat_y": (41, 1, 37),
          "flat_z": (2, 40, 39), "voxel": (1, 1, 1)}  # z, y, x


def _cast(monkeypatch, ctx, X, vol, cams, poses, c4p, step, n, rows, cols, shared, **kw):
    monkeypatch.setenv("XRH_CELL_REUSE", "0" if shared else "1")
    buf = ctx.alloc(4 * n * rows * cols)
    X.line_int(ctx, vol, cams, poses_f32(poses), c4p, step, buf, **kw)
    out = buf.download(np.float32).reshape(n, rows, cols)
    buf.free()
    return out


@pytest.mark.parametrize("kernel,geom", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("spacing", [0.6, 1.5, 4.0])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_slabs_equal_shared_rays(ctx, oracle, shape, spacing, kernel, geom, monkeypatch):
    from xreg_amd import _xrh as X
    from xreg_amd import geometry as G
    from xreg_amd import synth

    print(f"case: slabs {shape} spacing {spacing} kernel {kernel} geom {geom}", flush=True)
    rng = np.random.default_rng(7)
    vox = rng.uniform(0.01, 0.05, SHAPES[shape]).astype(np.float32)
    size = vox.shape[::-1]
    sp = 2.0
    center = G.vol_center_phys(size, sp)
    gt = G.gt_pose(center, 510.0)
    rows, cols = 45, 37  # partial tiles
    cam = G.camera(1020.0, rows, cols, 2.0 * spacing * sp, 2.0 * spacing * sp)
    # axis-aligned, small rotations, and views from anywhere (main axes x, y and z, both ways)
    poses = np.concatenate([gt[None], synth.random_poses(gt, center, 3, 10.0, 5.0, seed=1),
                            synth.random_poses(gt, center, 8, 180.0, 5.0, seed=2)])
    n = len(poses)
    c4p = np.zeros(n, np.int64)
    vol = X.Volume(ctx, vox, G.idx_to_phys(sp))
    for step in (0.45 * sp, 1.7 * sp):
        kw = dict(kernel=kernel, geom=geom)
        a = _cast(monkeypatch, ctx, X, vol, [cam], poses, c4p, step, n, rows, cols, False, **kw)
        b = _cast(monkeypatch, ctx, X, vol, [cam], poses, c4p, step, n, rows, cols, True, **kw)
        assert np.array_equal(a, b), (step, int((a != b).sum()))
        if geom == 0:
            ref, _ = oracle.drr_f32(vox, G.idx_to_phys(sp), [cam], poses_f32(poses), step=step, kernel=kernel)
            assert drr_rel_err(a, ref).max() <= DRR_REL_TOL, step
    vol.close()


@pytest.mark.parametrize("objs", [2, 3])
def test_objects_by_slabs_equal_shared_rays(ctx, objs, monkeypatch):
    from xreg_amd import _xrh as X
    from xreg_amd import geometry as G
    from xreg_amd import synth

    print(f"case: slabs, {objs} objects", flush=True)
    rng = np.random.default_rng(3)
    sp, rows, cols = 2.0, 50, 50
    vols = [X.Volume(ctx, rng.uniform(0.01, 0.05, (40, 42 + 5 * k, 44)).astype(np.float32), G.idx_to_phys(sp))
            for k in range(objs)]
    cam = G.camera(1020.0, rows, cols, 4.0, 4.0)
    fixed = X.Fixed(ctx, rng.random((rows, cols), dtype=np.float32), X.XRH_SIM_NCC)
    center = G.vol_center_phys((44, 42, 40), sp)
    gt = G.gt_pose(center, 510.0)
    n = 3
    poses = synth.random_poses(gt, center, n * objs, 40.0, 10.0, seed=5).reshape(n, objs, 4, 4)
    ev = np.tile(np.arange(objs, dtype=np.int32), (n, 1))
    b = X.Batch(ctx, [X.make_view(v, fixed, cam, 0.9) for v in vols], max_items=n * objs, geom=X.XRH_GEOM_FP64)
    out = ctx.alloc(4 * n * rows * cols)
    got = []
    for reuse in (1, 0):
        b.set_drr_variant(reuse, 0, 8)
        sims = [b.eval_objects(ev, poses, drr=out) for _ in range(3)][-1]  # graph replays
        got.append((sims, out.download(np.float32)))
    assert got[0][1].max() > 0.0
    assert np.array_equal(got[0][1], got[1][1])
    assert np.array_equal(got[0][0], got[1][0])
    out.free()
    b.close()
    fixed.close()
    for v in vols:
        v.close()
