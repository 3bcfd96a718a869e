"""Plain voxels, which slabs march by, are kept while a context's budget has room and given back when an
allocation needs theirs: the budget allows what it allowed without them, they are not charged, and casts,
batches (graph replays, before and after), several objects and a batch evaluating in another thread keep their
values bit for bit."""
import threading

import numpy as np
import pytest

from tests.helpers import poses_f32

pytestmark = pytest.mark.gpu

SHAPE = (170, 161, 163)  # z, y, x: 75 MB of cells, 19 MB of plain voxels
PLAIN = 4 * 172 * 163 * 165


def _scene(spacing, n=36):
    from xreg_amd import geometry as G
    from xreg_amd import synth

    rng = np.random.default_rng(8)
    vox = (rng.uniform(0.01, 0.05, SHAPE) * (rng.uniform(size=SHAPE) < 0.8)).astype(np.float32)
    center = G.vol_center_phys(SHAPE[::-1], 1.0)
    gt = G.gt_pose(center, 510.0)
    rows, cols = 130, 117
    cam = G.camera(1020.0, rows, cols, 2.0 * spacing, 2.0 * spacing)
    # 72 tiles a pose: enough poses that whole rays are cast
    poses = np.concatenate([gt[None], synth.random_poses(gt, center, n - 1, 30.0, 5.0, seed=2)])
    return vox, G.idx_to_phys(1.0), cam, poses, rng.random((rows, cols), dtype=np.float32)


def _give_back(c, budget):
    """Takes all of the budget that is charged to no one."""
    c.alloc(budget - c.bytes_in_use()).free()


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("spacing", [0.5, 0.8, 1.3, 3.0])
@pytest.mark.parametrize("geom", [0, 1])
def test_same_values_with_and_without(ctx, storage, spacing, geom):
    from xreg_amd import _xrh as X

    print(f"case: plain voxels given back, storage {storage} spacing {spacing} geom {geom}", flush=True)
    vox, i2p, cam, poses, fixed = _scene(spacing)
    n, npx = len(poses), fixed.size
    budget = 1 << 30
    got = []

    def run(c, vol, b, buf):
        X.line_int(c, vol, [cam], poses_f32(poses), np.zeros(n, np.int64), 0.6, buf, geom=geom)
        cast = buf.download(np.float32)
        sims = [b.eval(np.zeros(n, np.int32), poses, drr=buf) for _ in range(2)]
        assert np.array_equal(sims[0], sims[1])
        drr = buf.download(np.float32)
        pairs = poses.reshape(n // 2, 2, 4, 4)
        osims = [b.eval_objects(np.tile(np.arange(2, dtype=np.int32), (n // 2, 1)), pairs, drr=buf) for _ in range(2)]
        assert np.array_equal(osims[0], osims[1])
        got.append((cast, sims[0], drr, osims[0], buf.download(np.float32)[: n // 2 * npx]))

    for c in (ctx, X.Context(0, hbm_budget_bytes=budget)):
        vol = X.Volume(c, vox, i2p, storage=storage)
        buf = c.alloc(4 * n * npx)
        fx = X.Fixed(c, fixed, X.XRH_SIM_NCC)
        b = X.Batch(c, [X.make_view(vol, fx, cam, 0.6)] * 2, max_items=n, geom=geom)
        run(c, vol, b, buf)
        if c is not ctx:
            used = c.bytes_in_use()
            _give_back(c, budget)
            assert c.bytes_in_use() == used
            run(c, vol, b, buf)
        for o in (b, fx, vol):
            o.close()
        buf.free()
        if c is not ctx:
            c.close()
    assert got[0][0].max() > 0.0
    for k in (1, 2):
        for a, b in zip(got[0], got[k]):
            assert np.array_equal(a, b), k


def test_budget_is_what_it_was(ctx):
    """A budget that holds a volume and the memory of its upload holds it still, whatever other volumes'
    plain voxels took, and refuses one byte more; bytes in use and a volume's bytes leave them out."""
    from xreg_amd import _xrh as X

    print("case: budget with plain voxels", flush=True)
    vox, i2p, cam, poses, _ = _scene(0.8)
    probe = X.Context(0, hbm_budget_bytes=2 << 30)
    base = probe.bytes_in_use()
    v = X.Volume(probe, vox, i2p)
    each = probe.bytes_in_use() - base
    assert v.nbytes <= each < v.nbytes + PLAIN
    v.close()
    assert probe.bytes_in_use() == base
    probe.close()
    budget = base + 3 * each + 4 * vox.size
    c = X.Context(0, hbm_budget_bytes=budget)
    vols = [X.Volume(c, vox, i2p) for _ in range(3)]
    assert c.bytes_in_use() == base + 3 * each
    rest = c.alloc(budget - c.bytes_in_use())
    with pytest.raises(X.XrhError):
        c.alloc(1)
    with pytest.raises(X.XrhError):
        X.Volume(c, vox, i2p)
    rest.free()
    for v in vols:
        v.close()
    assert c.bytes_in_use() == base
    c.close()


def test_not_counted_without_a_budget(ctx):
    """A server admits jobs by the bytes in use of a context that has no budget itself."""
    from xreg_amd import _xrh as X

    print("case: bytes in use without a budget", flush=True)
    vox, i2p, _, _, _ = _scene(0.8)
    used = ctx.bytes_in_use()
    v = X.Volume(ctx, vox, i2p)
    assert v.nbytes <= ctx.bytes_in_use() - used < v.nbytes + PLAIN
    v.close()
    assert ctx.bytes_in_use() == used


def test_given_back_while_another_thread_evaluates():
    from xreg_amd import _xrh as X

    print("case: plain voxels given back under an evaluating thread", flush=True)
    vox, i2p, cam, poses, fixed = _scene(0.8, n=16)
    budget = 1 << 30
    c = X.Context(0, hbm_budget_bytes=budget)
    fx = X.Fixed(c, fixed, X.XRH_SIM_NCC)
    iv = np.zeros(len(poses), np.int32)
    for _ in range(3):
        vol = X.Volume(c, vox, i2p)
        b = X.Batch(c, [X.make_view(vol, fx, cam, 0.6)], max_items=len(poses))
        b.set_options(use_graph=False, time_kernels=False)
        want = b.eval(iv, poses)
        started, bad = threading.Event(), []

        def evaluate():
            for _ in range(40):
                got = b.eval(iv, poses)
                started.set()
                if not np.array_equal(got, want):
                    bad.append(got)

        t = threading.Thread(target=evaluate)
        t.start()
        started.wait(60)
        for _ in range(5):
            _give_back(c, budget)
        t.join(60)
        assert not t.is_alive() and not bad
        b.close()
        vol.close()
    fx.close()
    c.close()
