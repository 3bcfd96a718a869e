"""How a DRR launch is planned (no GPU): slabs only where every volume has its plain voxels and the layout
allows them, and tuned variants kept apart by what the best variant turns on."""
import os
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
F32, F16 = 0, 1
LINEAR, QUAD, OCT, COEF, FACE, BRICK = 0, 1, 2, 3, 4, 5


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    from xreg_amd import build as B

    if not B.LIB.exists():
        B.build()
    exe = tmp_path_factory.mktemp("plan") / "drr_plan"
    res = subprocess.run([B.HIPCC, *B.COMMON, str(ROOT / "tests" / "cpp" / "drr_plan.hip"), f"-L{B.HERE}", "-lxrh",
                          f"-Wl,-rpath,{B.HERE}", "-o", str(exe)], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr

    def plan(*launches, env=None):
        """launches: dicts; returns (parts, slabs, lds, window, whole rays, key) of each."""
        args = []
        for l in launches:
            d = dict(storage=F32, layout=FACE, geom=1, spacing=0.8, mb=215, plain=1, tiles=50000, reuse=-1, objs=1)
            d.update(l)
            args += [str(d[k]) for k in ("storage", "layout", "geom", "spacing", "mb", "plain", "tiles", "reuse", "objs")]
        e = {k: v for k, v in os.environ.items() if k != "XRH_CELL_REUSE"}
        out = subprocess.run([str(exe), *args], capture_output=True, text=True, env=dict(e, **(env or {})), check=True)
        rows = []
        for line in out.stdout.splitlines():
            a, key = line.split("|")
            p = [int(v) for v in a.split()]
            rows.append((p[0], bool(p[1]), p[2], p[3], bool(p[4]), key.strip()))
        return rows

    return plan


@pytest.mark.parametrize("env", [None, {"XRH_CELL_REUSE": "1"}])
def test_slabs_need_plain_voxels(planner, env):
    ok = planner(dict(), dict(storage=F16, layout=OCT, spacing=1.2), env=env)
    assert all(r[1] and r[0] == 1 and r[2] > 0 for r in ok)
    no = planner(dict(plain=0), dict(storage=F16, layout=OCT, spacing=1.2, plain=0), dict(layout=BRICK), dict(layout=COEF),
                 dict(layout=QUAD), dict(layout=LINEAR), env=env)
    assert not any(r[1] for r in no)
    assert all(r[0] == 1 for r in no)


def test_gathering_launches(planner):
    # close rays of a launch that only gathers are shared by two up to 2048 tiles, as where slabs do not pay
    assert planner(dict(plain=0, spacing=0.5, tiles=1500))[0][0] == 2
    assert planner(dict(layout=BRICK, spacing=0.5, tiles=1500))[0][0] == 2
    # LDS held back only by launches that gather sparse rays over a volume larger than the caches
    rows = planner(dict(plain=0, spacing=0.9), dict(plain=0, spacing=1.2), dict(plain=0, spacing=3.0),
                   dict(plain=0, spacing=1.2, mb=26), dict(layout=QUAD, spacing=1.2), dict(spacing=0.0))
    assert [r[2] > 0 for r in rows] == [False, True, True, False, False, False]
    assert rows[2][2] > rows[1][2]
    # windows shorten with the distance of the rays
    w = [r[3] for r in planner(*[dict(plain=0, spacing=s) for s in (0.0, 0.3, 0.5, 0.7, 0.9, 2.0)])]
    assert w[0] == 16 and w == sorted(w, reverse=True) and w[-1] == 1


def test_tuned_variants_are_kept_apart(planner):
    """A variant tuned for close rays (shared) must not be taken by sparse rays or another volume, another
    number of objects or a launch that cannot go by slabs; nearly the same launch takes it."""
    base = planner(dict(tiles=546))[0][5]
    others = planner(dict(tiles=546, spacing=1.94), dict(tiles=546, mb=1700), dict(tiles=546, objs=2),
                     dict(tiles=546, plain=0), dict(tiles=546, geom=0), dict(tiles=5460))
    assert all(r[5] != base for r in others)
    assert planner(dict(tiles=547, spacing=0.81, mb=216))[0][5] == base


def test_whole_rays_reported_as_run(planner):
    """What the tuner reports of the default is what is run: 546 tiles are shared by two when close and
    taken whole when sparse."""
    rows = planner(dict(tiles=546, spacing=0.4), dict(tiles=546, spacing=1.94), dict(tiles=546, spacing=1.94, reuse=0),
                   dict(tiles=546, spacing=0.4, reuse=1))
    assert [r[4] for r in rows] == [False, True, False, True]
    assert all((r[0] == 1) == r[4] for r in rows)


def test_launches_of_the_slab_tests_take_slabs(planner):
    """The launches that test_gpu_drr_budget.py compares with and without plain voxels, and the forced choice
    that the slab tests make."""
    rows = planner(dict(tiles=1296, mb=75, spacing=0.8), dict(tiles=1296, mb=75, spacing=0.8, objs=2),
                   dict(tiles=2592, mb=75, spacing=1.3, geom=0))
    assert all(r[1] for r in rows)
    forced = planner(dict(tiles=30, mb=1, spacing=0.4, objs=2), dict(tiles=30, mb=1, spacing=3.2, objs=3, geom=0),
                     dict(tiles=30, mb=1, spacing=0.4, storage=F16, layout=OCT), env={"XRH_CELL_REUSE": "1"})
    assert all(r[1] for r in forced)
    shared = planner(dict(tiles=30, mb=1, spacing=0.4), env={"XRH_CELL_REUSE": "0"})
    assert not shared[0][1] and shared[0][0] == 4


def test_sparse_rays_of_small_launches(planner):
    """Few sparse FP32 rays are shared by four waves whose lanes keep in step, more by two; close ones
    keep the long window."""
    rows = planner(*[dict(tiles=t, spacing=s, geom=0) for t, s in ((64, 2.3), (100, 3.5), (200, 2.8), (72, 1.43), (256, 0.6))])
    assert [r[0] for r in rows] == [4, 4, 2, 4, 4]
    assert [r[3] for r in rows] == [4, 1, 16, 4, 16]
