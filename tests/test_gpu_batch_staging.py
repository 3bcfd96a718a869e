"""Batches of the sizes at which the set-up kernel's workgroups begin and end (8 items each, plan and
similarity items copied beside them): the same values as each item evaluated alone, through graph
replays whose poses change between them, and eagerly."""
import numpy as np
import pytest

from tests.helpers import poses_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metric", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 65])
def test_sizes(ctx, oracle, n, metric):
    from xreg_amd import _xrh as X
    from xreg_amd import geometry as G
    from xreg_amd import synth

    print(f"case: batch staging n {n} metric {metric}", flush=True)
    rng = np.random.default_rng(n)
    vox = (rng.uniform(size=(24, 28, 32)) * 0.04).astype(np.float32)
    center = G.vol_center_phys(vox.shape[::-1], 2.0)
    gt = G.gt_pose(center, 510.0)
    cam = G.camera(1020.0, 40, 50, 3.0, 3.0)
    poses = synth.random_poses(gt, center, n, 20.0, 5.0, seed=5)
    fixed, _ = oracle.drr_f32(vox, G.idx_to_phys(2.0), [cam], poses_f32(gt[None]), step=1.0)
    vol = X.Volume(ctx, vox, G.idx_to_phys(2.0))
    fx = X.Fixed(ctx, fixed[0], metric)
    b = X.Batch(ctx, [X.make_view(vol, fx, cam, 1.0)], max_items=70)
    iv = np.zeros(n, np.int32)
    alone = np.array([b.eval(iv[:1], p[None])[0] for p in poses])
    assert np.array_equal(b.eval(iv, poses), alone)
    assert np.array_equal(b.eval(iv, poses[::-1].copy()), alone[::-1])
    b.set_options(use_graph=False, time_kernels=True)
    assert np.array_equal(b.eval(iv, poses), alone)
    b.close()
    fx.close()
    vol.close()
