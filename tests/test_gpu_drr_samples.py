"""Single trilinear samples of the FP32 layouts against the interpolation in double: rays with a step
longer than their chord have one sample, at a position that is known to the last bit.

Bound: with M the largest corner (none negative) and u = 2^-24, a face's edge differences, their products'
sums, the difference between the edges and the face's value are rounded once each, at most u M: 4 u M in all
with their weights; the step along x adds two roundings: 6 u M. Over many samples the error is also no larger
than that of a face written as c0 + c1 v + c2 w + c3 v w with c3 formed in double and rounded once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def _positions(cam, pose, size):
    """(x, y, z) of the only sample per pixel, float32 in the padded grid (voxel k at k + 1), NaN where the
    ray misses: the FP64 ray set-up with an identity index-to-physical transform."""
    kinv = np.array(cam.intrins_inv[:], np.float32).astype(np.float64).reshape(3, 3)
    einv = np.array(cam.extrins_inv[:], np.float32).astype(np.float64).reshape(4, 4)
    pin = np.array(cam.pinhole[:], np.float32).astype(np.float64)
    z = -float(np.float32(cam.focal_len))
    c, r = np.meshgrid(np.arange(cam.num_det_cols, dtype=np.float64), np.arange(cam.num_det_rows, dtype=np.float64))
    q = [z * c, z * r, np.full_like(c, z)]
    p = [(kinv[k, 0] * q[0] + kinv[k, 1] * q[1]) + kinv[k, 2] * q[2] for k in range(3)]
    det = [(einv[k, 0] * p[0] + einv[k, 1] * p[1]) + einv[k, 2] * p[2] + einv[k, 3] for k in range(3)]

    def point(v):
        return [(pose[k, 0] * v[0] + pose[k, 1] * v[1]) + pose[k, 2] * v[2] + pose[k, 3] for k in range(3)]

    ph, dp = point(pin), point(det)
    d = [dp[k] - ph[k] for k in range(3)]
    t0, t1 = np.zeros_like(c), np.ones_like(c)
    for k in range(3):
        a, b = (0.0 - ph[k]) * (1.0 / d[k]), (size[k] - 1 - ph[k]) * (1.0 / d[k])
        t0, t1 = np.maximum(t0, np.minimum(a, b)), np.minimum(t1, np.maximum(a, b))
    ok = (t1 - t0) > 2.0e-3
    pos = np.stack([((ph[k] + (t0 + 1.0e-3) * d[k]) + 1.0).astype(np.float32) for k in range(3)])
    return np.where(ok, pos, np.float32(np.nan))


def _fma(a, b, c):
    return (a.astype(np.float64) * b + c).astype(np.float32)


@pytest.mark.parametrize("layout", ["LAYOUT_FACE", "LAYOUT_BRICK"])
@pytest.mark.parametrize("content", ["random", "edges", "smooth"])
def test_one_sample(ctx, content, layout):
    from xreg_amd import _xrh as X
    from xreg_amd import geometry as G
    from xreg_amd import synth

    print(f"case: single samples {content} {layout}", flush=True)
    rng = np.random.default_rng(5)
    shape = (61, 66, 70)  # z, y, x
    if content == "random":
        vox = rng.random(shape)
    elif content == "edges":  # soft tissue, bone and air, voxel by voxel
        vox = rng.choice([0.0, 0.02, 0.05], shape) * (1.0 + 0.1 * rng.uniform(-1, 1, shape))
    else:
        vox = 0.02 * (1.0 + 0.04 * rng.uniform(-1, 1, shape))
    vox = vox.astype(np.float32)
    size = shape[::-1]
    center = G.vol_center_phys(size, 1.0)
    gt = G.gt_pose(center, 510.0)
    cam = G.camera(1020.0, 96, 96, 1.4, 1.4)
    poses = synth.random_poses(gt, center, 12, 180.0, 5.0, seed=9)
    poses = poses.astype(np.float32).astype(np.float64)  # (what line_int takes)
    n, step = len(poses), 256.0  # (a power of two: the scaled value is the sample)
    vol = X.Volume(ctx, vox, G.idx_to_phys(1.0), layout=getattr(X, layout))
    buf = ctx.alloc(4 * n * 96 * 96)
    X.line_int(ctx, vol, [cam], poses.reshape(n, 16), np.zeros(n, np.int64), step, buf, geom=X.XRH_GEOM_FP64)
    got = (buf.download(np.float32).reshape(n, 96, 96) / np.float32(step)).astype(np.float64)
    buf.free()
    vol.close()
    err, err4 = [], []
    pad = np.pad(vox, 1, mode="edge")
    for k in range(n):
        pos = _positions(cam, poses[k], size)
        hit = np.isfinite(pos[0])
        p = pos[:, hit]
        assert hit.sum() > 1000
        base = np.floor(p).astype(int)
        w = (p - base).astype(np.float32)
        v = np.stack([pad[base[2] + dz, base[1] + dy, base[0] + dx] for dz in (0, 1) for dy in (0, 1) for dx in (0, 1)])
        wx, wy, wz = w.astype(np.float64)
        e = v.astype(np.float64)
        ex = [e[2 * i] * (1 - wx) + e[2 * i + 1] * wx for i in range(4)]
        ey = [ex[2 * i] * (1 - wy) + ex[2 * i + 1] * wy for i in range(2)]
        want = ey[0] * (1 - wz) + ey[1] * wz
        d = got[k][hit] - want
        assert np.all(np.abs(d) <= 6.0 * U * v.max(axis=0)), float((np.abs(d) / v.max(axis=0)).max() / U)
        face = []
        for x in (0, 1):
            v00, v10, v01, v11 = v[x], v[2 + x], v[4 + x], v[6 + x]
            c3 = ((e[6 + x] - e[4 + x]) - (e[2 + x] - e[x])).astype(np.float32)
            face.append(_fma(w[2], _fma(w[1], c3, v01 - v00), _fma(w[1], v10 - v00, v00)))
        four = _fma(w[0], face[1], _fma(-w[0], face[0], face[0]))
        err.append(d)
        err4.append(four - want)
    rms = [float(np.sqrt(np.mean(np.concatenate(x) ** 2))) for x in (err, err4)]
    assert rms[0] <= rms[1], rms
