"""The band order of DRR workgroups: every tile of every item is cast exactly once whatever the
number of bands, on detectors with fewer tiles than bands, with one tile row, and with tile
counts that no band count divides."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,n", [(2, 2, 1), (16, 16, 11), (17, 33, 11), (5, 160, 3), (96, 96, 13),
                                         (113, 77, 1), (113, 77, 9)])
def test_bands_cover_every_tile_once(ctx, rows, cols, n):
    from xreg_amd import _xrh as X
    from xreg_amd import geometry as G
    from xreg_amd import synth

    print(f"case: bands {rows}x{cols} n={n}", flush=True)
    w = synth.config("c1", n_poses=n, small=True)
    cam = G.camera(1020.0, rows, cols, 240.0 / rows, 240.0 / cols)
    vol = X.Volume(ctx, w.vol, w.idx_to_phys)
    fixed = X.Fixed(ctx, np.random.default_rng(1).random((rows, cols), dtype=np.float32), X.XRH_SIM_NCC)
    b = X.Batch(ctx, [X.make_view(vol, fixed, cam, w.step)], max_items=n)
    out = ctx.alloc(4 * n * rows * cols)
    iv = np.zeros(n, np.int32)

    def cast(bands):
        out.upload(np.full(n * rows * cols, -1.0, np.float32))  # a tile left out would keep this
        b.set_drr_variant(1, 0, bands)
        sims = b.eval(iv, w.poses, drr=out)
        return out.download(np.float32), sims

    ref, ref_sims = cast(1)
    assert (ref >= 0.0).all() and ref.max() > 0.0
    for bands in (2, 3, 7, 8, 16):
        drr, sims = cast(bands)
        assert np.array_equal(drr, ref), bands
        assert np.array_equal(sims, ref_sims), bands
    out.free()
    b.close()
    fixed.close()
    vol.close()
