"""Slab marching over 16-bit volumes: the same DRRs bit for bit as rays gathered by several waves, for
rays close (which gather), a voxel and several voxels apart, SUM and MAX and both ray set-ups, on a volume large
enough to be taken by slabs; and the CPU reference's on the rounded voxels."""
import numpy as np
import pytest

from tests.helpers import DRR_REL_TOL, drr_rel_err, poses_f32

pytestmark = pytest.mark.gpu

SHAPE = (158, 163, 171)  # z, y, x: 4.4e6 voxels, 70 MB of cells


@pytest.fixture(scope="module")
def volumes(ctx):
    import torch

    from xreg_amd import _xrh as X
    from xreg_amd import geometry as G

    rng = np.random.default_rng(11)
    vox = (rng.uniform(0.01, 0.05, SHAPE) * (rng.uniform(size=SHAPE) < 0.7)).astype(np.float32)
    vols, rounded = {}, {}
    for storage, t in ((1, torch.float16), (2, torch.bfloat16)):
        vols[storage] = X.Volume(ctx, vox, G.idx_to_phys(1.0), storage=storage)
        rounded[storage] = torch.from_numpy(vox).to(t).to(torch.float32).numpy()
    yield vols, rounded
    for v in vols.values():
        v.close()


@pytest.mark.parametrize("kernel,geom", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("spacing", [0.2, 0.8, 3.0])
@pytest.mark.parametrize("storage", [1, 2])
def test_slabs_equal_shared_rays(ctx, oracle, volumes, storage, spacing, kernel, geom, monkeypatch):
    from xreg_amd import _xrh as X
    from xreg_amd import geometry as G
    from xreg_amd import synth

    print(f"case: 16-bit slabs storage {storage} spacing {spacing} kernel {kernel} geom {geom}", flush=True)
    vols, rounded = volumes
    center = G.vol_center_phys(SHAPE[::-1], 1.0)
    gt = G.gt_pose(center, 510.0)
    rows, cols = 45, 37
    cam = G.camera(1020.0, rows, cols, 2.0 * spacing, 2.0 * spacing)
    poses = np.concatenate([gt[None], synth.random_poses(gt, center, 5, 180.0, 5.0, seed=2)])
    n = len(poses)
    got = []
    for shared in ("1", "0"):
        monkeypatch.setenv("XRH_CELL_REUSE", shared)
        buf = ctx.alloc(4 * n * rows * cols)
        X.line_int(ctx, vols[storage], [cam], poses_f32(poses), np.zeros(n, np.int64), 0.6, buf, kernel=kernel, geom=geom)
        got.append(buf.download(np.float32).reshape(n, rows, cols))
        buf.free()
    assert np.array_equal(got[0], got[1])
    if geom == 0:
        ref, _ = oracle.drr_f32(rounded[storage], G.idx_to_phys(1.0), [cam], poses_f32(poses), step=0.6, kernel=kernel)
        assert drr_rel_err(got[0], ref).max() <= DRR_REL_TOL
