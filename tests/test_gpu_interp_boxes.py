"""The many-tap interpolators with rays at different distances, so that the taps' box of a wave's next
samples fits the workgroup's memory whole, at half the samples or not at all, on a detector that is no
multiple of a wave's 8 x 8 pixels, against the oracle; per pixel within the interpolators' 1e-4."""
import numpy as np
import pytest

from tests.helpers import DRR_REL_TOL, drr_rel_err, poses_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("interp", [2, 3])
@pytest.mark.parametrize("px,step", [(0.6, 0.9), (4.0, 0.9), (9.0, 2.5), (40.0, 7.0)])  # mm; voxels are 2 mm
@pytest.mark.parametrize("kernel,aa", [(0, 0), (1, 0), (0, 2)])
def test_ray_distances(ctx, oracle, interp, px, step, kernel, aa):
    from xreg_amd import _xrh as X
    from xreg_amd import geometry as G
    from xreg_amd import synth

    print(f"case: interp boxes interp {interp} px {px} step {step} kernel {kernel} aa {aa}", flush=True)
    rng = np.random.default_rng(int(10 * px))
    vox = (rng.uniform(size=(23, 30, 37)) * 0.04).astype(np.float32)
    sp = 2.0
    center = G.vol_center_phys(vox.shape[::-1], sp)
    gt = G.gt_pose(center, 510.0)
    cam = G.camera(1020.0, 21, 27, px, px)
    poses = poses_f32(np.concatenate([gt[None], synth.random_poses(gt, center, 2, 180.0, 6.0, seed=4)]))
    n = len(poses)
    vol = X.Volume(ctx, vox, G.idx_to_phys(sp))
    buf = ctx.alloc(4 * n * 21 * 27)
    X.line_int_interp(ctx, vol, [cam], poses, np.zeros(n, np.int64), step, buf, interp, kernel=kernel, aa_rays=aa,
                      aa_seed=7)
    got = buf.download(np.float32).reshape(n, cam.num_det_rows, cam.num_det_cols)
    buf.free()
    vol.close()
    ref, _ = oracle.drr_f32(vox, G.idx_to_phys(sp), [cam], poses, step=step, kernel=kernel, interp=interp, aa_rays=aa,
                            aa_seed=7)
    assert ref.max() > 0.0
    assert drr_rel_err(got, ref).max() <= DRR_REL_TOL
