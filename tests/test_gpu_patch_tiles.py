"""The patch kernels compiled for a diameter, masked and unmasked, against the general patch kernel
(which also writes the per-patch scores) at the edges of their 16 x 16 tiles of patches, and with a
NaN or an infinity in the moving image. Both form FP64 box sums and a FP32 result: they agree to the
rounding of that result (a few units of 6e-8; values lie in 0 .. 2)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metric", [2, 3])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("radius", [2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("patches", [(1, 1), (16, 17), (15, 33), (40, 16)])  # patch rows, columns
def test_against_general_kernel(ctx, metric, masked, radius, patches):
    from xreg_amd import _xrh as X

    print(f"case: patch tiles metric {metric} masked {masked} radius {radius} patches {patches}", flush=True)
    rows, cols = patches[0] + 2 * radius, patches[1] + 2 * radius
    rng = np.random.default_rng(radius + 10 * metric + 100 * patches[1])
    y, x = np.mgrid[0:rows, 0:cols]
    base = np.sin(x / 5.0) + np.cos(y / 7.0)
    fixed = (base + 0.05 * rng.standard_normal((rows, cols))).astype(np.float32)
    mov = (base[None] + 0.2 * rng.standard_normal((5, rows, cols))).astype(np.float32)
    mov[1] = 0.75  # no deviation anywhere
    mov[2, rows // 2, cols // 3] = np.nan
    mov[3, rows // 3, cols // 2] = np.inf
    mask = None
    if masked:
        mask = (rng.uniform(size=(rows, cols)) < 0.8).astype(np.uint8)
        mask[: rows // 3, : cols // 3] = 0
        mask[rows // 2, cols // 2] = 1
    fx = X.Fixed(ctx, fixed, metric, smooth_ksize=3, patch_radius=radius, patch_stride=1, mask=mask)
    buf = ctx.alloc(mov.nbytes)
    buf.upload(mov)
    got = fx.compute(buf, len(mov))
    want, _ = fx.patch_scores(buf, len(mov))
    buf.free()
    fx.close()
    assert np.isfinite(got[[0, 1, 4]]).all()
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert np.allclose(got[ok], want[ok], rtol=0.0, atol=1e-6)
