"""The workspace that downsampling keeps: charged to no one, kept by no context with a budget, and of each
thread's own when several downsample at once."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _image(seed, shape=(384, 401)):
    return np.random.default_rng(seed).random(shape, dtype=np.float32)


def test_bytes_in_use(ctx):
    from xreg_amd import _xrh as X

    print("case: pyramid workspace, bytes in use", flush=True)
    img = _image(1)
    used = ctx.bytes_in_use()
    want = X.downsample_image(ctx, img, 0.5)
    assert ctx.bytes_in_use() == used
    h, w = want.shape
    need = 2 * 8 * img.size + 4 * h * w + 4096  # two planes of doubles, the output and the weights
    budget = 32 << 20
    c = X.Context(0, hbm_budget_bytes=budget)
    base = c.bytes_in_use()
    for _ in range(2):
        assert np.array_equal(X.downsample_image(c, img, 0.5), want)
        assert c.bytes_in_use() == base
    # what fitted the budget before a call fits it after
    b = c.alloc(budget - base)
    with pytest.raises(X.XrhError):
        X.downsample_image(c, img, 0.5)
    b.free()
    b = c.alloc(budget - base - need)
    assert np.array_equal(X.downsample_image(c, img, 0.5), want)
    b.free()
    c.close()


def test_two_threads(ctx):
    from xreg_amd import _xrh as X

    print("case: pyramid workspace, two threads", flush=True)
    imgs = [_image(k, (200 + 40 * k, 300 - 30 * k)) for k in range(2)]
    want = [X.downsample_image(ctx, im, 0.5) for im in imgs]
    bad = []

    def run(k):
        for _ in range(25):
            if not np.array_equal(X.downsample_image(ctx, imgs[k], 0.5), want[k]):
                bad.append(k)

    threads = [threading.Thread(target=run, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not any(t.is_alive() for t in threads) and not bad
