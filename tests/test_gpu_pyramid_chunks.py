"""The chunked B-spline filter of xrh_downsample_image at its edges: lines shorter than the start
sum's horizon, of one to three samples, and around multiples of the row (256) and column (32)
chunks. The filter runs in double and the result is rounded to float once, so it lies within one
float unit in the last place of the image's maximum of the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 300), (300, 1), (2, 3), (3, 2), (17, 18), (19, 20), (31, 255),
                                       (32, 256), (33, 257), (34, 258), (63, 511), (64, 512), (65, 513), (97, 289)])
@pytest.mark.parametrize("factor", [0.5, 1.0])
def test_chunk_edges(ctx, oracle, rows, cols, factor):
    from xreg_amd import _xrh as X

    if int(rows * factor + 0.5) < 1 or int(cols * factor + 0.5) < 1:
        pytest.skip("empty output")
    print(f"case: pyramid chunks {rows}x{cols} factor {factor}", flush=True)
    img = np.random.default_rng(rows * 1000 + cols).random((rows, cols), dtype=np.float32)
    want = oracle.downsample_image(img, factor)
    for _ in range(2):  # the workspace is reused
        got = X.downsample_image(ctx, img, factor)
        assert got.shape == want.shape
        assert np.abs(got.astype(np.float64) - want).max() <= 2.0 ** -23 * max(1.0, float(np.abs(want).max()))
