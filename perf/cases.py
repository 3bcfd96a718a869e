"""Performance cases: the work a 2D/3D registration program has this framework do, through the
public Python entry points (xreg_amd._xrh).

Kinds of cases
  generation  one optimiser evaluation: n candidate poses x V views cast and scored in one batched
              submission (Batch.eval, FP64 ray set-up); n = 1 is a refiner's step
  objects     the same with several rigid objects per candidate, cast onto static background
              images (Batch.eval_objects)
  cast        the ray caster alone, as RayCaster::compute is called (line_int): either ray set-up,
              line sums or maximum-intensity projections, with or without background images
  score       a similarity metric alone on moving images that are in device memory
              (Fixed.compute), with masks, strides and patch sizes
  interp      casts with the other volume interpolators or anti-aliasing (line_int_interp)
  pyramid     fixed-image downsampling for one level of a multi-resolution registration
              (downsample_image, host image in and out)
  ingest      a Hounsfield CT volume in host memory made resident and its first projection cast

Volumes are ellipsoid phantoms in air (soft tissue, a cortical shell, a trabecular core) with
noise in the tissue; fixed images are projections at a pose near the candidates with detector
noise; poses are spread as a CMA-ES population or a refiner spreads them.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from xreg_amd import _xrh as X

FOCAL = 1020.0
STORAGE = {"f32": X.XRH_F32, "f16": X.XRH_F16, "bf16": X.XRH_BF16}
GEOM = {"fp32": X.XRH_GEOM_FP32, "fp64": X.XRH_GEOM_FP64}
METRIC = {"ncc": X.XRH_SIM_NCC, "grad_ncc": X.XRH_SIM_GRAD_NCC, "patch_ncc": X.XRH_SIM_PATCH_NCC,
          "patch_grad_ncc": X.XRH_SIM_PATCH_GRAD_NCC}
INTERP = {"linear": X.XRH_INTERP_LINEAR, "nn": X.XRH_INTERP_NN, "sinc": X.XRH_INTERP_SINC,
          "bspline": X.XRH_INTERP_BSPLINE}
BLUR = {0: [1.0], 3: [0.25, 0.5, 0.25], 5: [0.0625, 0.25, 0.375, 0.25, 0.0625],
        7: [0.03125, 0.109375, 0.21875, 0.28125, 0.21875, 0.109375, 0.03125]}
# HUToLinAtt's default attenuation constants (1/mm)
MU_WATER, MU_AIR, HU_LOWER = 0.02683, 0.02485e-4, -1000.0


# ------------------------------------------------------------------------------------------
# the cases

def _geometry(size, spacing, rows, cols, px, step, **more):
    return dict(vx=size[0], vy=size[1], vz=size[2], spacing=spacing, rows=rows, cols=cols, px=px, step=step, **more)


C1 = ((128, 128, 96), 2.0)
C2 = ((256, 256, 200), 1.0)
C4 = ((512, 512, 400), 0.5)


def listed():
    return [
        # the smallest call: one pose of a refiner at the coarse level of a small volume
        dict(name="refine_192_ncc", kind="generation", n=1, views=1, storage="f32", metric="ncc", smooth=0, radius=5,
             rot=1.0, trans=2.0, **_geometry(*C1, 192, 192, 1.552, 1.0)),
        # a refiner's step at the fine level: one pose, the default patch metric
        dict(name="refine_384_patch", kind="generation", n=1, views=1, storage="f32", metric="patch_grad_ncc",
             smooth=5, radius=5, rot=1.0, trans=2.0, **_geometry(*C2, 384, 384, 0.776, 0.5)),
        # the coarse level of a three-view registration: 50 candidates x 3 views on 96^2 detectors
        dict(name="cmaes_3view_96", kind="generation", n=50, views=3, storage="f32", metric="grad_ncc", smooth=5,
             radius=5, rot=10.0, trans=15.0, **_geometry(*C2, 96, 96, 3.104, 0.5)),
        # the headline: a CMA-ES generation of 100 candidates, single view, patch gradient-NCC
        dict(name="cmaes_384", kind="generation", n=100, views=1, storage="f32", metric="patch_grad_ncc", smooth=5,
             radius=5, rot=10.0, trans=15.0, **_geometry(*C2, 384, 384, 0.776, 0.5)),
        # full-resolution volume and detector, FP32 and 16-bit storage (the largest work)
        dict(name="cmaes_768_f32", kind="generation", n=16, views=1, storage="f32", metric="ncc", smooth=0, radius=5,
             rot=8.0, trans=10.0, **_geometry(*C4, 768, 768, 0.388, 0.25)),
        dict(name="cmaes_768_f16", kind="generation", n=16, views=1, storage="f16", metric="patch_ncc", smooth=0,
             radius=5, rot=8.0, trans=10.0, **_geometry(*C4, 768, 768, 0.388, 0.25)),
        # two bones moving on their own in front of a static background (pelvis and femur)
        dict(name="two_objects_256", kind="objects", n=30, views=1, objs=2, storage="f32", metric="grad_ncc", smooth=5,
             radius=5, rot=5.0, trans=8.0, **_geometry((192, 192, 192), 1.5, 256, 256, 1.164, 0.75)),
        # the drop-in caster with the reference's float arithmetic on a cropped, odd-sized detector
        dict(name="cast_fp32_odd", kind="cast", n=24, views=1, storage="f32", geom="fp32", op="sum", bg=False,
             rot=10.0, trans=15.0, **_geometry((185, 201, 173), 1.3, 331, 277, 0.9, 0.8)),
        # the patch metric with the collimator masked out
        dict(name="score_masked_384", kind="score", n=20, metric="patch_grad_ncc", smooth=5, radius=5, stride=1,
             mask=True, rows=384, cols=384),
        # projections with the B-spline interpolator (simulated studies)
        dict(name="interp_bspline_192", kind="interp", n=4, views=1, storage="f32", interp="bspline", aa=0, op="sum",
             rot=10.0, trans=15.0, **_geometry(*C1, 192, 192, 1.552, 1.0)),
        # a fixed image brought to a quarter of its size for the coarse level
        dict(name="pyramid_768_quarter", kind="pyramid", rows=768, cols=768, factor=0.25),
        # a new CT volume and its first projection
        dict(name="ingest_256", kind="ingest", n=1, views=1, storage="f32", rot=5.0, trans=5.0,
             **_geometry(*C2, 192, 192, 1.552, 1.0)),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_geometry(rng, dmin, dmax):
    m = rng.uniform(96, 512)
    size = [max(64, min(512, int(m * rng.uniform(0.75, 1.0)))) for _ in range(3)]
    spacing = round(256.0 / max(size) * rng.uniform(0.9, 1.3), 3)
    cols = _log_int(rng, dmin, dmax)
    rows = max(dmin, min(dmax, int(cols * rng.uniform(0.7, 1.3))))
    return _geometry(size, spacing, rows, cols, round(298.0 / max(rows, cols), 4),
                     round(spacing * rng.uniform(0.4, 0.8), 4))


def _cap(case, cap):
    """Fewer poses where a case would cost more than the largest listed one."""
    per = case["rows"] * case["cols"] * case["vy"] * case["spacing"] / case["step"] * case.get("objs", 1)
    case["n"] = max(1, min(case["n"], int(cap / (per * case["views"]))))
    return case


def draw(rng):
    kind = rng.choice(["generation"] * 5 + ["cast"] * 2 + ["score"] * 2 + ["objects", "interp", "pyramid", "ingest"])
    if kind == "generation":
        return _cap(dict(kind=kind, n=_log_int(rng, 1, 100), views=rng.choice([1, 1, 2, 3]),
                         storage=rng.choice(["f32", "f32", "f16", "bf16"]), metric=rng.choice(list(METRIC)),
                         smooth=rng.choice([0, 3, 5, 7]), radius=rng.choice([3, 4, 5, 5, 6]),
                         rot=rng.choice([1.0, 5.0, 10.0]), trans=rng.choice([2.0, 15.0]),
                         **_draw_geometry(rng, 64, 768)), 6.0e9)
    if kind == "objects":
        return _cap(dict(kind=kind, n=_log_int(rng, 2, 40), views=1, objs=rng.choice([2, 3]), storage="f32",
                         metric=rng.choice(["ncc", "grad_ncc", "patch_grad_ncc"]), smooth=5, radius=5, rot=5.0,
                         trans=8.0, **_draw_geometry(rng, 96, 384)), 3.0e9)
    if kind == "cast":
        return _cap(dict(kind=kind, n=_log_int(rng, 1, 60), views=rng.choice([1, 2]),
                         storage=rng.choice(["f32", "f16", "bf16"]), geom=rng.choice(["fp32", "fp64"]),
                         op=rng.choice(["sum", "sum", "max"]), bg=rng.choice([False, True]), rot=10.0, trans=15.0,
                         **_draw_geometry(rng, 64, 768)), 4.0e9)
    if kind == "score":
        cols = _log_int(rng, 64, 768)
        rows = max(48, int(cols * rng.uniform(0.7, 1.3)))
        n = max(1, min(_log_int(rng, 1, 100), int(6.0e6 / (rows * cols))))
        return dict(kind=kind, n=n, metric=rng.choice(list(METRIC)), smooth=rng.choice([0, 3, 5, 7]),
                    radius=rng.choice([3, 5, 5, 8]), stride=rng.choice([1, 1, 2]), mask=rng.choice([False, True]),
                    rows=rows, cols=cols)
    if kind == "interp":
        how = rng.choice(["bspline", "sinc", "nn", "linear"])
        aa = rng.choice([2, 4]) if how == "linear" else rng.choice([0, 0, 4]) if how == "nn" else 0
        return _cap(dict(kind=kind, n=_log_int(rng, 1, 6), views=1, storage="f32", interp=how, aa=aa,
                         op=rng.choice(["sum", "max"]), rot=10.0, trans=15.0, **_draw_geometry(rng, 64, 192)),
                    3.0e7)
    if kind == "pyramid":
        cols = _log_int(rng, 96, 1024)
        return dict(kind=kind, rows=max(64, int(cols * rng.uniform(0.7, 1.3))), cols=cols,
                    factor=rng.choice([0.5, 0.25, 0.125]))
    g = _draw_geometry(rng, 64, 256)
    return dict(kind="ingest", n=1, views=1, storage=rng.choice(["f32", "f32", "f16"]), rot=5.0, trans=5.0, **g)


# ------------------------------------------------------------------------------------------
# inputs, from the seed alone

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _phantom(case, seed):
    """Attenuation voxels (z, y, x) on the GPU, float32."""
    dim = (case["vx"], case["vy"], case["vz"])
    rng = np.random.default_rng(seed)
    ax = [torch.arange(n, device="cuda", dtype=torch.float32) - (n - 1) / 2.0 for n in dim]

    def radius(fracs, shrink=0.0):
        q = [(ax[k] / (fracs[k] * dim[k] - shrink)) ** 2 for k in range(3)]
        return q[2][:, None, None] + q[1][None, :, None] + q[0][None, None, :]

    body, bone = rng.uniform(0.42, 0.46, 3), rng.uniform(0.27, 0.31, 3)
    vol = torch.zeros(dim[2], dim[1], dim[0], device="cuda")
    noise = torch.empty_like(vol).uniform_(-0.1, 0.1, generator=_gen(seed))
    vol = torch.where(radius(body) <= 1.0, 0.02 * (1.0 + 0.4 * noise), vol)
    vol = torch.where(radius(bone) <= 1.0, 0.05 * (1.0 + 0.3 * noise), vol)
    return torch.where(radius(bone, 2.0) <= 1.0, 0.03 * (1.0 + noise), vol)


def _center(case):
    return case["spacing"] * np.array([case["vx"], case["vy"], case["vz"]], dtype=np.float64) / 2.0


def _index_to_phys(case):
    m = np.eye(4, dtype=np.float32)
    m[0, 0] = m[1, 1] = m[2, 2] = np.float32(case["spacing"])
    return m


def _rigid(R, t):
    T = np.eye(4)
    T[:3, :3], T[:3, 3] = R, t
    return T


def _euler(a):
    (cx, cy, cz), (sx, sy, sz) = np.cos(a), np.sin(a)
    rx = np.array([[1, 0, 0], [0, cx, -sx], [0, sx, cx]])
    ry = np.array([[cy, 0, sy], [0, 1, 0], [-sy, 0, cy]])
    rz = np.array([[cz, -sz, 0], [sz, cz, 0], [0, 0, 1]])
    return rz @ ry @ rx


def _true_pose(case):
    """Camera to physical: an antero-posterior view, the volume's centre at the isocentre."""
    ap = np.array([[1.0, 0.0, 0.0], [0.0, 0.0, -1.0], [0.0, 1.0, 0.0]])
    return _rigid(np.eye(3), _center(case)) @ _rigid(ap, (0, 0, 0)) @ _rigid(np.eye(3), (0, 0, FOCAL / 2.0))


def _poses(case, seed, count):
    rng = np.random.default_rng(seed + 1)
    c = _center(case)
    out = np.empty((count, 4, 4))
    for i in range(count):
        R = _euler(np.deg2rad(rng.normal(0.0, case["rot"], 3)))
        out[i] = _rigid(np.eye(3), c) @ _rigid(R, rng.normal(0.0, case["trans"], 3)) @ _rigid(np.eye(3), -c) @ \
            _true_pose(case)
    return out


def _cameras(case):
    """(inverse intrinsics, inverse extrinsics) per view, float32: detector along camera -z, views
    30 degrees apart about the isocentre."""
    k = np.array([[-FOCAL / case["px"], 0, (case["cols"] - 1) / 2.0], [0, -FOCAL / case["px"], (case["rows"] - 1) / 2.0],
                  [0, 0, 1]])
    iso = FOCAL / 2.0
    out = []
    for v in range(case["views"]):
        R = _euler(np.array([0.0, np.deg2rad(30.0 * v), 0.0]))
        E = _rigid(np.eye(3), (0, 0, -iso)) @ _rigid(R, (0, 0, 0)) @ _rigid(np.eye(3), (0, 0, iso))
        out.append((np.linalg.inv(k).astype(np.float32), E.astype(np.float32)))
    return out


def _camera_struct(case, kinv, einv):
    c = X.Camera()
    c.num_det_rows, c.num_det_cols, c.coord_frame, c.focal_len = case["rows"], case["cols"], 1, FOCAL
    c.intrins_inv[:] = [float(v) for v in kinv.reshape(-1)]
    c.extrins_inv[:] = [float(v) for v in einv.reshape(-1)]
    c.pinhole[:] = [float(v) for v in einv[:3, 3]]
    c.det_row_spacing = c.det_col_spacing = case["px"]
    return c


def _noisy(img, gen):
    return (img + torch.randn(img.shape, device="cuda", generator=gen, dtype=img.dtype) * (0.01 * img.max())).float()


def _fixed_images(case, seed, vols, backgrounds=None):
    """One fixed image per view: the projection at the true pose (every object there) with noise."""
    g = _gen(seed + 2)
    out = []
    for v, (kinv, einv) in enumerate(_cameras(case)):
        img = sum(_line_integral(case, vol, kinv, einv, _true_pose(case), step=2.0 * case["step"]) for vol in vols)
        if backgrounds is not None:
            img = img + backgrounds[v].double()
        out.append(_noisy(img, g))
    return out


def _smooth_images(n, rows, cols, seed):
    """Projection-like images: broad bright shapes with edges and noise, float32 on the GPU."""
    g = _gen(seed + 3)
    y = torch.linspace(-1, 1, rows, device="cuda")[:, None]
    x = torch.linspace(-1, 1, cols, device="cuda")[None, :]
    p = torch.empty(n, 6, 6, device="cuda").uniform_(0.0, 1.0, generator=g)
    img = torch.zeros(n, rows, cols, device="cuda")
    for k in range(6):
        a = [p[:, k, j, None, None] for j in range(6)]
        q = ((x - (a[0] - 0.5)) / (0.2 + 0.8 * a[1])) ** 2 + ((y - (a[2] - 0.5)) / (0.2 + 0.8 * a[3])) ** 2
        img += (0.5 + a[4]) * torch.sqrt(torch.clamp(1.0 - q, min=0.0))
    return img + 0.02 * torch.randn(img.shape, device="cuda", generator=g)


def _moving_images(case, seed):
    """Moving images that correlate with the fixed one as candidates near the optimum do."""
    base = _smooth_images(1, case["rows"], case["cols"], seed)
    other = _smooth_images(case["n"], case["rows"], case["cols"], seed + 100)
    fixed = base[0] + 0.02 * torch.randn(base[0].shape, device="cuda", generator=_gen(seed + 4))
    return fixed.contiguous(), (0.7 * base + 0.3 * other).contiguous()


def _mask(case):
    """A collimator: a disc of unmasked pixels, and a blocked corner inside it."""
    y, x = np.mgrid[0:case["rows"], 0:case["cols"]]
    r = ((x / (case["cols"] - 1) - 0.5) / 0.48) ** 2 + ((y / (case["rows"] - 1) - 0.5) / 0.48) ** 2
    m = (r <= 1.0).astype(np.uint8)
    m[: case["rows"] // 5, : case["cols"] // 4] = 0
    return m


def _background(case, seed):
    return [im for im in _smooth_images(case["views"], case["rows"], case["cols"], seed + 5)]


def _hu(case, seed):
    """Hounsfield units of the phantom (air -1000), float32."""
    mu = _phantom(case, seed)
    return (mu - MU_WATER) * (1000.0 / (MU_WATER - MU_AIR))


# ------------------------------------------------------------------------------------------
# the state a program holds

class _Device:
    """A torch tensor's memory as the framework's entry points take device buffers."""

    def __init__(self, tensor):
        self.tensor, self.ptr, self.nbytes = tensor, tensor.data_ptr(), tensor.numel() * tensor.element_size()


class State(dict):
    """What a program keeps between calls; framework objects are closed with it."""

    def __del__(self):
        try:
            _context().synchronize()
            for key in ("batch", "fixed", "vols"):
                for obj in self.get(key, ()):
                    obj.close()
        except Exception:
            pass


_CONTEXT = []


def _context():
    if not _CONTEXT:
        _CONTEXT.append(X.Context(0))
    return _CONTEXT[0]


def prepare(case, seed):
    ctx = _context()
    s = State(case=case, kind=case["kind"], ctx=ctx)
    kind = case["kind"]
    if kind == "pyramid":
        img = _smooth_images(1, case["rows"], case["cols"], seed)[0]
        s["img"] = np.ascontiguousarray(img.cpu().numpy())
        return s
    if kind == "score":
        fixed, mov = _moving_images(case, seed)
        s["fixed"] = [X.Fixed(ctx, fixed.cpu().numpy(), METRIC[case["metric"]], smooth_ksize=case["smooth"],
                              patch_radius=case["radius"], patch_stride=case["stride"],
                              mask=_mask(case) if case["mask"] else None)]
        s["mov"] = _Device(mov)
        torch.cuda.synchronize()
        return s
    s["cams"] = [_camera_struct(case, *kv) for kv in _cameras(case)]
    npix = case["rows"] * case["cols"]
    if kind == "ingest":
        s["hu"] = np.ascontiguousarray(_hu(case, seed).cpu().numpy())
        s["i2p"] = _index_to_phys(case)
        s["poses"] = _poses(case, seed, 1)
        s["drr"] = _Device(torch.zeros(1, case["rows"], case["cols"], device="cuda"))
        torch.cuda.synchronize()
        return s
    objs = case.get("objs", 1)
    mu = [_phantom(case, seed + 1000 * k) for k in range(objs)]
    s["vols"] = [X.Volume(ctx, m.cpu().numpy(), _index_to_phys(case), storage=STORAGE[case["storage"]]) for m in mu]
    items = case["n"] * case["views"]
    s["drr"] = _Device(torch.zeros(items, case["rows"], case["cols"], device="cuda"))
    if kind in ("cast", "interp"):
        # view-major projections, as the caster distributes poses among camera models
        s["poses"] = np.tile(_poses(case, seed, case["n"]), (case["views"], 1, 1)).astype(np.float32)
        s["cam_for_proj"] = np.repeat(np.arange(case["views"], dtype=np.int64), case["n"])
        if case.get("bg"):
            s["bg"] = _Device(torch.stack(_background(case, seed)).contiguous())
        torch.cuda.synchronize()
        return s
    bg = _background(case, seed) if kind == "objects" else None
    fixed = [f.cpu().numpy() for f in _fixed_images(case, seed, mu, bg)]
    s["fixed"] = [X.Fixed(ctx, f, METRIC[case["metric"]], smooth_ksize=case["smooth"], patch_radius=case["radius"])
                  for f in fixed]
    if kind == "objects":
        views = [X.make_view(v, s["fixed"][0], s["cams"][0], case["step"]) for v in s["vols"]]
        s["bg"] = _Device(torch.stack(bg * objs).contiguous())
        s["entry_view"] = np.tile(np.arange(objs, dtype=np.int32), (case["n"], 1))
        s["entry_pose"] = _poses(case, seed, case["n"] * objs).reshape(case["n"], objs, 4, 4)
        s["batch"] = [X.Batch(ctx, views, case["n"] * objs, geom=X.XRH_GEOM_FP64)]
    else:
        views = [X.make_view(s["vols"][0], f, c, case["step"]) for f, c in zip(s["fixed"], s["cams"])]
        s["item_view"] = np.repeat(np.arange(case["views"], dtype=np.int32), case["n"])
        s["item_pose"] = np.tile(_poses(case, seed, case["n"]), (case["views"], 1, 1))
        s["batch"] = [X.Batch(ctx, views, items, geom=X.XRH_GEOM_FP64)]
    torch.cuda.synchronize()
    return s


def run(state):
    case, kind, ctx = state["case"], state["kind"], state["ctx"]
    if kind == "generation":
        sims = state["batch"][0].eval(state["item_view"], state["item_pose"], drr=state["drr"])
        return {"sims": sims, "drr": state["drr"].tensor}
    if kind == "objects":
        sims = state["batch"][0].eval_objects(state["entry_view"], state["entry_pose"], bg=state["bg"],
                                              drr=state["drr"])
        return {"sims": sims, "drr": state["drr"].tensor}
    if kind == "cast":
        X.line_int(ctx, state["vols"][0], state["cams"], state["poses"], state["cam_for_proj"], case["step"],
                   state["drr"], kernel=X.XRH_LINE_INT_MAX if case["op"] == "max" else X.XRH_LINE_INT_SUM,
                   bg=state.get("bg"), geom=GEOM[case["geom"]])
        return {"drr": state["drr"].tensor}
    if kind == "score":
        return {"sims": state["fixed"][0].compute(state["mov"], case["n"])}
    if kind == "interp":
        X.line_int_interp(ctx, state["vols"][0], state["cams"], state["poses"], state["cam_for_proj"], case["step"],
                          state["drr"], INTERP[case["interp"]],
                          kernel=X.XRH_LINE_INT_MAX if case["op"] == "max" else X.XRH_LINE_INT_SUM,
                          aa_rays=case["aa"], aa_seed=7)
        return {"drr": state["drr"].tensor}
    if kind == "pyramid":
        return {"img": X.downsample_image(ctx, state["img"], case["factor"])}
    vol = X.Volume(ctx, state["hu"], state["i2p"], storage=STORAGE[case["storage"]], hu={})
    X.line_int(ctx, vol, state["cams"], state["poses"], np.zeros(1, np.int64), case["step"], state["drr"],
               geom=X.XRH_GEOM_FP64)
    vol.close()
    return {"drr": state["drr"].tensor}


# ------------------------------------------------------------------------------------------
# what a pass cannot do without

def _tissue_samples(case):
    """Samples of one projection that lie in tissue, from the true pose's chords through the body."""
    kinv, einv = _cameras(case)[0]
    det, ph = _detector(case, kinv, einv)
    p = _true_pose(case)
    det, ph = det @ p[:3, :3].T + p[:3, 3], p[:3, :3] @ ph + p[:3, 3]
    axes = 0.44 * case["spacing"] * np.array([case["vx"], case["vy"], case["vz"]])
    d = (det - ph)
    length = np.linalg.norm(d, axis=1)
    u, o = d / axes, (ph - _center(case)) / axes
    a, b, c = (u * u).sum(1), u @ o, float(o @ o) - 1.0
    disc = np.maximum(b * b - a * c, 0.0)
    return float((2.0 * np.sqrt(disc) / a * length / case["step"]).sum())


def work(case):
    if case["kind"] == "pyramid":
        n = case["rows"] * case["cols"]
        out = round(case["rows"] * case["factor"]) * round(case["cols"] * case["factor"])
        # two separable smoothing passes, two recursive filter passes, 16 taps per output pixel
        taps = 2 * int(4.0 * 0.5 / case["factor"]) + 1
        return {"bytes": 4.0 * (n + out), "flops": n * (4.0 * taps + 12.0) + 40.0 * out}
    npix = case["rows"] * case["cols"]
    if case["kind"] == "score":
        per_pixel = {"ncc": 6.0, "grad_ncc": 60.0, "patch_ncc": 40.0, "patch_grad_ncc": 120.0}[case["metric"]]
        images = {"ncc": 1, "grad_ncc": 2, "patch_ncc": 1, "patch_grad_ncc": 2}[case["metric"]]
        return {"bytes": 4.0 * npix * (case["n"] + images), "flops": per_pixel * npix * case["n"]}
    casts = case["n"] * case["views"] * case.get("objs", 1)
    samples = casts * _tissue_samples(case) * max(1, case.get("aa", 0))
    voxels = case["vx"] * case["vy"] * case["vz"] * case.get("objs", 1)
    width = 4 if case["storage"] == "f32" else 2
    images = case["n"] * case["views"] + (case["views"] if case["kind"] in ("generation", "objects") else 0)
    # a trilinear sample: the position, seven interpolations and the sum
    flops = {"bspline": 160.0, "sinc": 1170.0, "nn": 4.0}.get(case.get("interp"), 24.0)
    return {"bytes": voxels * (4.0 if case["kind"] == "ingest" else width) + 4.0 * npix * images,
            "flops": samples * flops}


# ------------------------------------------------------------------------------------------
# the same values in 64 bits

def _detector(case, kinv, einv):
    """Detector points (rows * cols, 3) and the focal point in camera-world coordinates."""
    r, c = np.mgrid[0:case["rows"], 0:case["cols"]]
    q = -FOCAL * np.stack([c.ravel(), r.ravel(), np.ones(r.size)], axis=1).astype(np.float64)
    k, e = kinv.astype(np.float64), einv.astype(np.float64)
    return (q @ k.T) @ e[:3, :3].T + e[:3, 3], e[:3, 3]


def _rays(case, kinv, einv, pose, step):
    """Start, step vector (index units) and last sample index (-1: miss) per pixel, on the GPU."""
    det, ph = _detector(case, kinv, einv)
    v = det - ph
    m = np.linalg.inv(_index_to_phys(case).astype(np.float64)) @ pose
    d = torch.from_numpy(v @ m[:3, :3].T).cuda()
    o = torch.from_numpy(m[:3, :3] @ ph + m[:3, 3]).cuda()
    hi = torch.tensor([case["vx"] - 1.0, case["vy"] - 1.0, case["vz"] - 1.0], dtype=torch.float64, device="cuda")
    flat = d.abs() <= 1.0e-8
    safe = torch.where(flat, torch.ones_like(d), d)
    a, b = (0.0 - o) / safe, (hi - o) / safe
    lo, up = torch.minimum(a, b), torch.maximum(a, b)
    lo = torch.where(flat, torch.full_like(lo, -math.inf), lo).amax(1).clamp(min=0.0)
    up = torch.where(flat, torch.full_like(up, math.inf), up).amin(1).clamp(max=1.0)
    ok = ~(flat & ((o < 0.0) | (o > hi))).any(1) & (up - lo > 2.0e-3)
    lo, up = lo + 1.0e-3, up - 1.0e-3
    dlen = d.norm(dim=1)
    s = torch.from_numpy(np.linalg.norm((v / np.linalg.norm(v, axis=1, keepdims=True) * float(np.float32(step)))
                                        @ m[:3, :3].T, axis=1)).cuda()
    n = torch.where(ok, torch.floor((up - lo) * dlen / s), torch.full_like(s, -1.0))
    return o + lo[:, None] * d, d * (s / dlen)[:, None], n


def _cast(case, sampler, kinv, einv, pose, step=None, op="sum"):
    """One projection in 64 bits: sampler(points (..., 3)) gives the volume's samples."""
    step = case["step"] if step is None else step
    start, d, n = _rays(case, kinv, einv, pose, step)
    hit = torch.nonzero(n >= 0)[:, 0]
    img = torch.zeros(n.numel(), dtype=torch.float64, device="cuda")
    if hit.numel():
        start, d, last = start[hit], d[hit], n[hit]
        acc = torch.zeros_like(last) if op == "sum" else torch.full_like(last, -math.inf)
        chunk = max(1, int(4.0e6 // hit.numel()))
        total = int(last.max().item()) + 1
        for i0 in range(0, total, chunk):
            i = torch.arange(i0, min(total, i0 + chunk), dtype=torch.float64, device="cuda")
            f = sampler(start[:, None, :] + i[None, :, None] * d[:, None, :])
            inside = i[None, :] <= last[:, None]
            if op == "sum":
                acc += torch.where(inside, f, torch.zeros_like(f)).sum(1)
            else:
                acc = torch.maximum(acc, torch.where(inside, f, torch.full_like(f, -math.inf)).amax(1))
        img[hit] = acc * float(np.float32(step))
    if op == "max":
        # a ray that misses leaves the background (0)
        img = torch.clamp(img, min=0.0)
    return img.reshape(case["rows"], case["cols"])


def _linear_sampler(vol):
    v = vol.double()[None, None]
    size = torch.tensor([vol.shape[2] - 1.0, vol.shape[1] - 1.0, vol.shape[0] - 1.0], dtype=torch.float64,
                        device="cuda")

    def sample(p):
        g = (p * (2.0 / size) - 1.0)[None, None]
        return torch.nn.functional.grid_sample(v, g, mode="bilinear", padding_mode="border",
                                               align_corners=True)[0, 0, 0]

    return sample


def _line_integral(case, vol, kinv, einv, pose, step=None, op="sum"):
    return _cast(case, _linear_sampler(vol), kinv, einv, pose, step, op)


def _spline_coefficients(vol):
    """Cubic B-spline coefficients with mirror boundaries: the collocation system per axis."""
    c = vol.double()
    for axis in range(3):
        n = c.shape[axis]
        a = torch.zeros(n, n, dtype=torch.float64, device="cuda")
        k = torch.arange(n, device="cuda")
        a[k, k] = 4.0 / 6.0
        a[k[1:], k[:-1]] += 1.0 / 6.0
        a[k[:-1], k[1:]] += 1.0 / 6.0
        a[0, 1] += 1.0 / 6.0
        a[n - 1, n - 2] += 1.0 / 6.0
        c = torch.linalg.solve(a, c.movedim(axis, 0).reshape(n, -1)).reshape(c.movedim(axis, 0).shape).movedim(0, axis)
    return c.contiguous()


def _tap_sampler(grid, taps, first, weights, mirror):
    """Separable interpolation over taps^3 voxels from floor(x) + first on."""
    dim = (grid.shape[2], grid.shape[1], grid.shape[0])
    flat = grid.reshape(-1)

    def sample(p):
        index, w = [], []
        for k in range(3):
            base = torch.floor(p[..., k])
            w.append(weights(p[..., k] - base))
            i = base.long()[..., None] + (torch.arange(taps, device="cuda") + first)
            if mirror:
                i = i.abs()
                i = torch.where(i > dim[k] - 1, 2 * (dim[k] - 1) - i, i)
            else:
                w[k] = torch.where((i >= 0) & (i < dim[k]), w[k], torch.zeros_like(w[k]))
                i = i.clamp(0, dim[k] - 1)
            index.append(i)
        out = torch.zeros(p.shape[:-1], dtype=torch.float64, device="cuda")
        for z in range(taps):
            for y in range(taps):
                row = (index[2][..., z] * dim[1] + index[1][..., y]) * dim[0]
                v = (flat[row[..., None] + index[0]] * w[0]).sum(-1)
                out += v * w[1][..., y] * w[2][..., z]
        return out

    return sample


def _bspline_weights(t):
    u = 1.0 - t
    return torch.stack([u ** 3 / 6.0, 2.0 / 3.0 - t * t + 0.5 * t ** 3, 2.0 / 3.0 - u * u + 0.5 * u ** 3, t ** 3 / 6.0],
                       dim=-1)


def _lanczos_weights(t):
    x = t[..., None] + (3.0 - torch.arange(8, dtype=torch.float64, device="cuda"))
    return torch.sinc(x) * torch.sinc(x / 4.0)


def _gradients(img, smooth):
    """Sobel x and y of (n, rows, cols) after the optional blur, mirrored at the border pixel."""
    def correlate(a, taps, axis):
        r = len(taps) // 2
        pad = (r, r, 0, 0) if axis == 2 else (0, 0, r, r)
        p = torch.nn.functional.pad(a[:, None], pad, mode="reflect")[:, 0] if r else a
        size = a.shape[axis]
        return sum(w * p.narrow(axis, k, size) for k, w in enumerate(taps))

    taps = BLUR[smooth]
    s = correlate(correlate(img, taps, 2), taps, 1)
    return (correlate(correlate(s, [-1.0, 0.0, 1.0], 2), [1.0, 2.0, 1.0], 1),
            correlate(correlate(s, [1.0, 2.0, 1.0], 2), [-1.0, 0.0, 1.0], 1))


def _ncc(f, m, mask):
    keep = torch.ones_like(f, dtype=torch.bool) if mask is None else mask
    fv, mv = f[keep], m[:, keep]
    n = fv.numel()
    fz, mz = fv - fv.mean(), mv - mv.mean(1, keepdim=True)
    sf = torch.sqrt(fz.square().sum() / (n - 1)).clamp(min=1.0e-6)
    sm = torch.sqrt(mz.square().sum(1) / (n - 1)).clamp(min=1.0e-6)
    return (1.0 - (mz @ fz) / (n * sf * sm)) * 0.5


def _patch(f, m, mask, radius, stride):
    d = 2 * radius + 1

    def box(a):
        rows = sum(a[..., k:a.shape[-2] - d + 1 + k, :] for k in range(d))
        return sum(rows[..., k:a.shape[-1] - d + 1 + k] for k in range(d))[..., ::stride, ::stride]

    n = float(d * d)
    k = torch.ones_like(f) if mask is None else mask.double()
    mu_f, cnt = box(f) / n, box(k)
    sd_f = torch.sqrt(((box(f * f) - n * mu_f * mu_f) / (n - 1.0)).clamp(min=0.0)).clamp(min=1.0e-6)
    w = torch.ones_like(cnt) if mask is None else cnt / cnt.sum()
    # patches of next to no weight are left out of the sum, not of its divisor
    used, total = torch.where(w.abs() > 1.0e-6, w, torch.zeros_like(w)), w.sum()
    out = []
    for a in m:
        a = a - a.mean()
        mu = box(a) / n
        sd = torch.sqrt(((box(a * a) - n * mu * mu) / (n - 1.0)).clamp(min=0.0)).clamp(min=1.0e-6)
        cross = box(a * f * k) - mu_f * box(a * k) - mu * box(f * k) + mu * mu_f * cnt
        out.append((used * (1.0 - cross / (sd * sd_f * n))).sum() / total)
    return torch.stack(out)


def _similarity(case, fixed, mov, mask=None):
    """The metric's values of (n, rows, cols) moving images against a fixed image."""
    f, m = fixed.double(), mov.double()
    f = f - f.mean()
    k = None if mask is None else torch.from_numpy(mask.astype(bool)).cuda()
    radius, stride = case["radius"], case.get("stride", 1)
    if case["metric"] == "ncc":
        return _ncc(f, m, k)
    if case["metric"] == "patch_ncc":
        return _patch(f, m, k, radius, stride)
    out = []
    fx, fy = (g[0] for g in _gradients(f[None], case["smooth"]))
    for a in m:
        gx, gy = _gradients(a[None], case["smooth"])
        one = _ncc if case["metric"] == "grad_ncc" else (lambda p, q, r: _patch(p, q, r, radius, stride))
        out.append(0.5 * (one(fx, gx, k) + one(fy, gy, k))[0])
    return torch.stack(out)


def _bessel_kernel(variance):
    """The discrete Gaussian e^-t I_n(t) truncated at 99% of its mass and normalised, from the
    polynomial approximations of I0 and I1 (Abramowitz and Stegun 9.8.1-9.8.4) and the recurrence."""
    if variance < 3.75:
        q = (variance / 3.75) ** 2
        i0 = np.polyval([0.45813e-2, 0.360768e-1, 0.2659732, 1.2067492, 3.0899424, 3.5156229, 1.0], q)
        i1 = variance * np.polyval([0.32411e-3, 0.301532e-2, 0.2658733e-1, 0.15084934, 0.51498869, 0.87890594, 0.5], q)
    else:
        q, s = 3.75 / variance, math.exp(variance) / math.sqrt(variance)
        i0 = s * np.polyval([0.392377e-2, -0.1647633e-1, 0.2635537e-1, -0.2057706e-1, 0.916281e-2, -0.157565e-2,
                             0.225319e-2, 0.1328592e-1, 0.39894228], q)
        i1 = s * np.polyval([-0.420059e-2, 0.1787654e-1, -0.2895312e-1, 0.2282967e-1, -0.1031555e-1, 0.163801e-2,
                             -0.362018e-2, -0.3988024e-1, 0.39894228], q)
    half = [math.exp(-variance) * i0, math.exp(-variance) * i1]
    total = half[0] + 2.0 * half[1]
    while total < 0.99:
        i = len(half)
        half.append(half[i - 2] - 2.0 * (i - 1) / variance * half[i - 1])
        total += 2.0 * half[i]
        if half[i] <= 0.0 or len(half) > 32:
            break
    h = np.array(half) / total
    return np.concatenate([h[:0:-1], h])


def _downsample(img, factor):
    taps = _bessel_kernel((0.5 / factor) ** 2)
    r = len(taps) // 2
    a = img.astype(np.float64)
    for axis in (1, 0):
        p = np.pad(a, [(r, r) if k == axis else (0, 0) for k in range(2)], mode="edge")
        n = a.shape[axis]
        a = sum(w * np.take(p, np.arange(n) + k, axis=axis) for k, w in enumerate(taps))
    a = a.astype(np.float32).astype(np.float64)
    out = a
    for axis in (0, 1):
        n, m = img.shape[axis], int(img.shape[axis] * factor + 0.5)
        k = np.arange(n)
        c = np.zeros((n, n))
        c[k, k] = 4.0 / 6.0
        c[k[1:], k[:-1]] += 1.0 / 6.0
        c[k[:-1], k[1:]] += 1.0 / 6.0
        c[0, 1] += 1.0 / 6.0
        c[n - 1, n - 2] += 1.0 / 6.0
        x = np.arange(m) / factor
        base, w = np.floor(x).astype(int), np.zeros((m, n))
        t = x - base
        u = 1.0 - t
        for j, v in enumerate((u ** 3 / 6, 2 / 3 - t * t + t ** 3 / 2, 2 / 3 - u * u + u ** 3 / 2, t ** 3 / 6)):
            i = np.abs(base - 1 + j)
            i = np.where(i > n - 1, 2 * (n - 1) - i, i)
            np.add.at(w, (np.arange(m), i), v)
        out = np.moveaxis(np.tensordot(w @ np.linalg.inv(c), out, axes=(1, axis)), 0, axis)
    return out


def _stored(vol, storage):
    return vol if storage == "f32" else vol.half().float() if storage == "f16" else vol.bfloat16().float()


def exact(case, seed):
    kind = case["kind"]
    if kind == "pyramid":
        return {"img": _downsample(_smooth_images(1, case["rows"], case["cols"], seed)[0].cpu().numpy(), case["factor"])}
    if kind == "score":
        fixed, mov = _moving_images(case, seed)
        return {"sims": _similarity(case, fixed, mov, _mask(case) if case["mask"] else None)}
    cams = _cameras(case)
    if kind == "ingest":
        mu = (_hu(case, seed).double() * ((MU_WATER - MU_AIR) * 1.0e-3) + MU_WATER -
              (HU_LOWER * (MU_WATER - MU_AIR) * 1.0e-3 + MU_WATER)).clamp(min=0.0)
        vol = _stored(mu.float(), case["storage"])
        pose = _poses(case, seed, 1)[0].astype(np.float32).astype(np.float64)
        return {"drr": _line_integral(case, vol, *cams[0], pose)[None]}
    mu = [_phantom(case, seed + 1000 * k) for k in range(case.get("objs", 1))]
    vols = [_stored(m, case["storage"]) for m in mu]
    if kind in ("cast", "interp"):
        if case.get("aa", 0) or case.get("interp") == "nn":
            return None  # jittered rays, and lookups that turn on the last bit of a position
        if case.get("interp") == "bspline":
            sampler = _tap_sampler(_spline_coefficients(vols[0]), 4, -1, _bspline_weights, True)
        elif case.get("interp") == "sinc":
            sampler = _tap_sampler(vols[0].double(), 8, -3, _lanczos_weights, False)
        else:
            sampler = _linear_sampler(vols[0])
        poses = _poses(case, seed, case["n"]).astype(np.float32).astype(np.float64)
        drr = torch.stack([_cast(case, sampler, *c, p, op=case["op"]) for c in cams for p in poses])
        if case.get("bg"):
            bg = torch.stack(_background(case, seed)).double().repeat_interleave(case["n"], 0)
            drr = bg + drr if case["op"] == "sum" else torch.maximum(bg, drr)
        return {"drr": drr}
    bg = _background(case, seed) if kind == "objects" else None
    fixed = _fixed_images(case, seed, mu, bg)
    samplers = [_linear_sampler(v) for v in vols]
    sims, drrs = [], []
    poses = _poses(case, seed, case["n"] * len(vols)).reshape(case["n"], len(vols), 4, 4)
    for v, c in enumerate(cams):
        drr = torch.stack([sum(_cast(case, s, *c, p) for s, p in zip(samplers, ps)) for ps in poses])
        if bg is not None:
            drr = drr + bg[v].double()
        sims.append(_similarity(case, fixed[v], drr))
        drrs.append(drr)
    return {"sims": torch.cat(sims), "drr": torch.cat(drrs)}
