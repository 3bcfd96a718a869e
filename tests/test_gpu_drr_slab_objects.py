"""Several objects per item cast by the slab kernel, which uses its boxes and corner tables again for each
object: the same DRRs and fused NCC values as rays shared by waves, for two and three objects that lie in
different places and move on their own (other boxes per object, one of them beside the detector), FP32 and
16-bit storage, SUM and MAX, both set-ups, through graph replays. (tests/test_drr_plan.py holds the launches
that take slabs; the forced choice takes them whatever the sizes.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel,geom", [(0, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("storage", [0, 1])
@pytest.mark.parametrize("spacing", [0.4, 1.2, 3.2])
@pytest.mark.parametrize("objs", [2, 3])
def test_objects_by_slabs(ctx, objs, spacing, storage, kernel, geom, monkeypatch):
    from xreg_amd import _xrh as X
    from xreg_amd import geometry as G
    from xreg_amd import synth

    print(f"case: slab objects {objs} spacing {spacing} storage {storage} kernel {kernel} geom {geom}", flush=True)
    rng = np.random.default_rng(3)
    rows, cols = 66, 83
    shapes = [(60, 62, 64), (41, 50, 39), (70, 33, 52)][:objs]
    vols = [X.Volume(ctx, rng.uniform(0.01, 0.05, s).astype(np.float32), G.idx_to_phys(1.0), storage=storage)
            for s in shapes]
    cam = G.camera(1020.0, rows, cols, 2.0 * spacing, 2.0 * spacing)
    fixed = X.Fixed(ctx, rng.random((rows, cols), dtype=np.float32), X.XRH_SIM_NCC)
    n = 4
    poses = np.empty((n, objs, 4, 4))
    for k, s in enumerate(shapes):
        center = G.vol_center_phys(s[::-1], 1.0)
        gt = G.gt_pose(center, 510.0)
        poses[:, k] = synth.random_poses(gt, center, n, 180.0, 12.0 * spacing, seed=5 + k)
    poses[-1, 0, :3, 3] += 4000.0  # off the detector
    ev = np.tile(np.arange(objs, dtype=np.int32), (n, 1))
    out = ctx.alloc(4 * n * rows * cols)
    got = []
    for reuse in ("1", "0"):
        monkeypatch.setenv("XRH_CELL_REUSE", reuse)
        b = X.Batch(ctx, [X.make_view(v, fixed, cam, 0.45, kernel=kernel) for v in vols], max_items=n * objs, geom=geom)
        sims = [b.eval_objects(ev, poses, drr=out) for _ in range(3)]
        assert all(np.array_equal(s, sims[0]) for s in sims[1:])
        got.append((sims[0], out.download(np.float32)))
        b.close()
    assert got[0][1].max() > 0.0
    assert np.array_equal(got[0][1], got[1][1])
    assert np.array_equal(got[0][0], got[1][0])
    out.free()
    fixed.close()
    for v in vols:
        v.close()
