"""Rays that begin at different depths: every way of marching (slabs, whole rays gathered, rays shared by
waves) sums the same samples by the same operations, so the DRRs are equal bit for bit, also where the lanes
of a wave enter tissue at different samples (scattered voxels and blobs in air, FP64 and FP32 set-up) and
under the bricked and the coefficient layouts."""
import numpy as np
import pytest

from tests.helpers import poses_f32

pytestmark = pytest.mark.gpu


BUDGET = 1 << 30


@pytest.fixture(scope="module")
def gather_ctx():
    """A context with a budget: taking all of it that is free makes its volumes give up their plain voxels,
    and whole rays gather then."""
    from xreg_amd import _xrh as X

    c = X.Context(0, hbm_budget_bytes=BUDGET)
    yield c
    c.close()


def _scattered(rng, shape, density):
    vox = np.zeros(shape, np.float32)
    on = rng.random(shape) < density
    vox[on] = rng.uniform(0.01, 0.05, int(on.sum()))
    z, y, x = np.ogrid[:shape[0], :shape[1], :shape[2]]
    for _ in range(5):
        c, r = [rng.integers(8, n - 8) for n in shape], rng.uniform(2, 8)
        ball = (z - c[0]) ** 2 + (y - c[1]) ** 2 + (x - c[2]) ** 2 <= r * r
        vox[ball] = 0.03 * (1.0 + 0.3 * rng.uniform(-1, 1, int(ball.sum())))
    return vox


@pytest.mark.parametrize("layout", ["face", "brick", "coef"])
@pytest.mark.parametrize("geom", [0, 1])
@pytest.mark.parametrize("spacing", [0.4, 0.6, 0.75, 0.95, 1.1, 1.8, 3.5])
def test_all_marches_equal(ctx, gather_ctx, monkeypatch, spacing, geom, layout):
    from xreg_amd import _xrh as X
    from xreg_amd import geometry as G
    from xreg_amd import synth

    print(f"case: march start, spacing {spacing} geom {geom} {layout}", flush=True)
    rng = np.random.default_rng(3)
    shape = (90, 101, 97)
    vox = _scattered(rng, shape, 2.0e-4)
    center = G.vol_center_phys(shape[::-1], 1.0)
    gt = G.gt_pose(center, 510.0)
    rows, cols = 70, 61
    cam = G.camera(1020.0, rows, cols, 2.0 * spacing, 2.0 * spacing)
    poses = synth.random_poses(gt, center, 8, 180.0, 8.0, seed=11)
    n = len(poses)
    got = []
    lay = {"face": X.LAYOUT_FACE, "brick": X.LAYOUT_BRICK, "coef": X.LAYOUT_COEF}[layout]
    for c, reuse in ((ctx, "1"), (gather_ctx, "1"), (ctx, "0"), (gather_ctx, "0")):
        monkeypatch.setenv("XRH_CELL_REUSE", reuse)
        vol = X.Volume(c, vox, G.idx_to_phys(1.0), layout=lay)
        if c is gather_ctx:
            c.alloc(BUDGET - c.bytes_in_use()).free()
        buf = c.alloc(4 * n * rows * cols)
        X.line_int(c, vol, [cam], poses_f32(poses), np.zeros(n, np.int64), 0.43, buf, geom=geom)
        got.append(buf.download(np.float32))
        buf.free()
        vol.close()
    assert got[0].max() > 0.0
    for k in (1, 2, 3):
        assert np.array_equal(got[0], got[k]), (k, int((got[0] != got[k]).sum()))
