"""Measured workloads of the cone-beam projector and its reconstruction passes.

Each case is one call (or the few calls of one solver step) through the
public entry points: ``gtt.capi.Context`` on device arrays, or a whole program
of ``gtt.operators`` on host arrays.  Scan geometries are the standard
workloads' (128^3 FDK, 256^3 ordered subsets, 512^3 with 720 views: voxel and
detector pitch give about 1.9 detector texels per voxel, SAD 1000 mm, SDD 1500
mm) and the uneven-scan distribution of the serving workload (edges of 96 to
320 voxels, detectors of 256 to 768 columns, neither a multiple of anything).

Inputs are a seeded phantom of ellipsoids (a body and ten inserts) as a scan
meets it: the volume sampled at voxel centres with a little texture, the
projections as exact line integrals with detector noise.

``exact`` evaluates the same passes in 64 bits with plain torch operations.
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "gt-tomography_amd"))

from gtt import capi  # noqa: E402
from gtt import operators as ops  # noqa: E402

SAD, SDD, SPP = 1000.0, 1500.0, 1.5
DEV = "cuda"


# ------------------------------------------------------------------- cases
def _scan(kind, n, views, nu, nv=None, nz=None, mm=None, arc=360.0, storage="f32", **more):
    """A case on an n x n x nz volume whose detector is 1.56 volume widths
    wide (the standard workloads' ratio) with square pixels."""
    return dict({"kind": kind, "n": n, "nz": n if nz is None else nz, "views": views, "nu": nu,
                 "nv": (3 * nu) // 4 if nv is None else nv, "mm": 1.0 if mm is None else mm, "arc": arc,
                 "storage": storage}, **more)


def listed():
    def case(name, *a, **k):
        return dict(_scan(*a, **k), name=name)
    return [
        # One ordered-subset step of a small volume (preview or test size):
        # project the subset, residual, backproject, update.  Launch and host
        # latency count most.
        case("sart_64", "sart", 64, 9, 96),
        # The forward projection of the 128^3 FDK workload, all views.
        case("fp_128", "fp", 128, 180, 256),
        # The whole FDK program at that size, host projections to host volume
        # (weights, ramp filter, FBP, projection of the result, rescale).
        case("fdk_128", "fdk", 128, 180, 256),
        # A volume lower than the detector's coverage (a region of interest
        # in z), so the outer rows' rays leave through its top and bottom.
        case("fp_slab_256", "fp", 256, 90, 512, nz=160, mm=0.8),
        # One subset step of the 256^3, 360-view, 10-subset workload.
        case("sart_256", "sart", 256, 36, 512, mm=0.8),
        # One subset step of a scan of the uneven batch (odd edge, ragged
        # detector), BF16 working copies as the server may be asked for.
        case("sart_291_bf16", "sart", 291, 32, 667, 500, storage="bf16"),
        # The image update of osMOMSolverD with TV (gradient step, two fused
        # TV proximal steps, momentum) at 256^3.
        case("mom_256", "mom", 256, 36, 512, mm=0.8),
        # The FDK pre-filter of the 512^3 workload's sinogram: 552,960 rows of
        # 1024, cosine weights and ramp filter.
        case("filter_1024", "filter", 512, 720, 1024, mm=0.5),
        # The 512^3, 720-view projector pair: backprojection and forward
        # projection with BF16 and with FP32 working copies; the FP32
        # backprojection with the FDK weight.
        case("bp_512_bf16", "bp", 512, 720, 1024, mm=0.5, storage="bf16", fbp=False),
        case("bp_512_fbp", "bp", 512, 720, 1024, mm=0.5, fbp=True),
        case("fp_512_bf16", "fp", 512, 720, 1024, mm=0.5, storage="bf16"),
        case("fp_512", "fp", 512, 720, 1024, mm=0.5),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed kinds: edges 48..448 and views 6..540
    (spread over their logarithm), detectors of 1.5 to 2.6 pixels per voxel,
    volumes from half as high as wide to cubes."""
    kind = rng.choice(["fp", "fp", "sart", "sart", "bp", "bp", "filter", "mom", "fdk"])
    n = _log_int(rng, 48, 192 if kind == "fdk" else 448)
    nu = int(n * rng.uniform(1.5, 2.6))
    nv = int(nu * rng.choice([0.75, 0.75, rng.uniform(0.6, 1.0)]))
    nz = n if rng.random() < 0.6 else int(n * rng.uniform(0.5, 1.0))
    views = {"sart": _log_int(rng, 6, 90), "fdk": _log_int(rng, 60, 360)}.get(kind, _log_int(rng, 12, 540))
    more = {"bp": {"fbp": rng.random() < 0.5},
            "filter": {"short": rng.random() < 0.3}}.get(kind, {})
    # a short scan covers half a turn
    arc = 180.0 if more.get("short") else 360.0
    storage = rng.choice(["f32", "bf16"]) if kind in ("fp", "bp", "sart") else "f32"
    return _scan(kind, n, views, nu, nv, nz, rng.choice([0.5, 0.8, 1.0]), arc, storage, **more)


# ------------------------------------------------------------------ inputs
def _geom(c):
    lxy, fu = c["n"] * c["mm"], 1.56 * c["n"] * c["mm"]
    return capi.Geom.make((c["n"], c["n"], c["nz"]), (lxy, lxy, c["nz"] * c["mm"]), (c["nu"], c["nv"]),
                          (fu, fu * c["nv"] / c["nu"]), SAD, SDD)


def _angles(c):
    return (np.arange(c["views"], dtype=np.float32) * np.float32(c["arc"] / c["views"])).astype(np.float32)


def _phantom(c, seed):
    """Ellipsoids as (centre, semi-axes, rotation about z, attenuation)."""
    rng = random.Random(seed)
    lxy, lz = c["n"] * c["mm"], c["nz"] * c["mm"]
    out = [((0.0, 0.0, 0.0), (0.42 * lxy, 0.36 * lxy, 0.47 * lz), 0.0, 0.02)]
    for _ in range(10):
        out.append((tuple(rng.uniform(-0.2, 0.2) * s for s in (lxy, lxy, lz)),
                    tuple(rng.uniform(0.03, 0.16) * s for s in (lxy, lxy, lz)),
                    rng.uniform(0.0, math.pi), rng.uniform(-0.01, 0.02)))
    return out


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _volume(c, seed):
    """(nz, n, n) attenuation per mm at the voxel centres, 1% texture."""
    ax = [((torch.arange(m, device=DEV) + 0.5) / m - 0.5) * (m * c["mm"]) for m in (c["n"], c["n"], c["nz"])]
    x, y, z = ax[0][None, None, :], ax[1][None, :, None], ax[2][:, None, None]
    vol = torch.randn((c["nz"], c["n"], c["n"]), device=DEV, generator=_generator(seed)).mul_(2e-4)
    for (cx, cy, cz), (a, b, d), rot, mu in _phantom(c, seed):
        co, si = math.cos(rot), math.sin(rot)
        xy = ((co * (x - cx) + si * (y - cy)) / a) ** 2 + ((co * (y - cy) - si * (x - cx)) / b) ** 2
        vol += mu * ((xy + ((z - cz) / d) ** 2) <= 1.0)
    return vol


def _projections(c, seed):
    """(views, nv, nu) line integrals of the phantom, with detector noise."""
    g, proj = _geom(c), torch.empty((c["views"], c["nv"], c["nu"]), device=DEV)
    u = ((torch.arange(g.nu, device=DEV) + 0.5) / g.nu - 0.5) * g.fov_u
    v = ((torch.arange(g.nv, device=DEV) + 0.5) / g.nv - 0.5) * g.fov_v
    u, v = u[None, :], v[:, None]
    shapes = _phantom(c, seed)
    for k, th in enumerate(np.deg2rad(_angles(c).astype(np.float64))):
        ct, st = math.cos(th), math.sin(th)
        p = torch.zeros((g.nv, g.nu), device=DEV)
        for (cx, cy, cz), axes, rot, mu in shapes:
            # the ray in the ellipsoid's frame, scaled to the unit sphere
            co, si = math.cos(rot + 0.0), math.sin(rot + 0.0)
            sx, sy = st * SAD - cx, -ct * SAD - cy
            dx, dy = ct * u - st * SDD, st * u + ct * SDD
            o = [(co * sx + si * sy) / axes[0], (co * sy - si * sx) / axes[1], -cz / axes[2]]
            d = [(co * dx + si * dy) / axes[0], (co * dy - si * dx) / axes[1], v / axes[2]]
            dd = d[0] ** 2 + d[1] ** 2 + d[2] ** 2
            od = o[0] * d[0] + o[1] * d[1] + o[2] * d[2]
            disc = od * od - dd * (o[0] ** 2 + o[1] ** 2 + o[2] ** 2 - 1.0)
            p += (2.0 * mu) * torch.sqrt(torch.clamp(disc, min=0.0)) / dd * torch.sqrt(u * u + v * v + SDD * SDD)
        proj[k] = p
    return proj.add_(torch.randn(proj.shape, device=DEV, generator=_generator(seed + 1)), alpha=0.01)


def _mom_inputs(c, seed):
    """Iterate, prox point, gradient image and preconditioner of one step."""
    x = _volume(c, seed)
    noise = torch.randn(x.shape, device=DEV, generator=_generator(seed + 2))
    return {"x": x, "xold": x + 5e-4 * noise, "z": x - 1e-3 * noise, "img": 30.0 * noise.flip(0),
            "precon": 1e-4 * (1.0 + 0.3 * torch.rand(x.shape, device=DEV, generator=_generator(seed + 3)))}


MOM = {"step": -1.0, "sigma": 1.0 / (16 * 1e-5), "tau": 1e-5, "weight": 1.0, "avg_lambda": 1e-3, "c": 0.6,
       "steps": 2}


def _inputs(c, seed):
    k = c["kind"]
    if k == "fp":
        return {"vol": _volume(c, seed)}
    if k in ("bp", "filter", "fdk"):
        return {"proj": _projections(c, seed)}
    if k == "mom":
        return _mom_inputs(c, seed)
    # sart: the measured subset, the current image (another phantom's, so the
    # residual is not noise alone), its normalisers
    n3 = (c["nz"], c["n"], c["n"])
    gen = _generator(seed + 4)
    return {"b": _projections(c, seed), "x": _volume(c, seed + 5).clamp_(min=0.0),
            "wp": 1.0 / (20.0 + 150.0 * torch.rand((c["views"], c["nv"], c["nu"]), device=DEV, generator=gen)),
            "wx": 1.0 / (c["views"] * (0.9 + 0.2 * torch.rand(n3, device=DEV, generator=gen)))}


def prepare(case, seed):
    g = _geom(case)
    s = dict(_inputs(case, seed), case=case, g=g)
    if case["kind"] == "fdk":
        s["proj"] = s["proj"].cpu().numpy()
        s["angles"] = _angles(case)
        s["filter"] = np.arange(g.nu + 1, dtype=np.float32)   # Ram-Lak
        return s
    ctx = s["ctx"] = capi.Context(torch.cuda.current_device())
    ctx.set_views(_angles(case))
    ctx.storage(case["storage"])
    if case["kind"] == "filter":
        ctx.set_filter(capi.default_filter(g.nu))
    if case["kind"] in ("fp", "sart"):
        s["out"] = torch.empty(g.proj_shape(case["views"]), device=DEV)
    elif case["kind"] == "filter":
        s["out"] = torch.empty_like(s["proj"])
    if case["kind"] in ("bp", "sart"):
        s["img"] = torch.empty(g.vol_shape, device=DEV)
    if case["kind"] == "mom":
        s["g"] = torch.empty(g.vol_shape, device=DEV)
    return s


# -------------------------------------------------------------------- runs
def run(state):
    case, g = state["case"], state["g"]
    kind = case["kind"]
    if kind == "fdk":
        vol, scale = ops.fdk_reconstruct_3d(g, state["angles"], None, state["proj"], filt=state["filter"])
        return {"vol": vol, "scale": scale}
    ctx = state["ctx"]
    if kind == "fp":
        return ctx.fp(g, state["vol"], state["out"], samples_per_pixel=SPP)
    if kind == "bp":
        return ctx.bp(g, state["proj"], state["img"], fbp=case["fbp"])
    if kind == "filter":
        return ctx.fdk_prefilter(g, state["proj"], state["out"], short_scan=case.get("short", False))
    if kind == "sart":
        # the subset step of OS-SART
        ctx.fp(g, state["x"], state["out"], samples_per_pixel=SPP)
        ctx.sart_residual(state["out"], state["b"], state["wp"])
        ctx.bp(g, state["out"], state["img"])
        ctx.sart_update(state["x"], state["img"], state["wx"], 1.0, True)
        return {"x": state["x"], "r": state["out"]}
    # mom: the image update of osMOMSolverD after a subset's backprojection
    x, t = state["x"], state["g"]
    tau, sigma = MOM["tau"], MOM["sigma"]
    ctx.mom_gradient_step(state["z"], state["img"], state["precon"], MOM["step"])
    for _ in range(MOM["steps"]):
        ctx.tv_update_g(x, t, state["z"], state["precon"], sigma, 0.0, MOM["weight"], tau, MOM["avg_lambda"])
        x, t = t, x
    ctx.mom_momentum(x, state["xold"], state["z"], MOM["c"], True)
    return {"x": x, "z": state["z"]}


def work(case):
    nvox = case["n"] ** 2 * case["nz"]
    nproj = case["nu"] * case["nv"] * case["views"]
    samples = nproj * int(SPP * case["n"])   # a lerp and an addition each
    updates = nvox * case["views"]           # three lerps and an addition each
    # two rows per transform of 2 nu points and its inverse
    fft = nproj / (2 * case["nu"]) * 2 * 5 * (2 * case["nu"]) * math.log2(2 * case["nu"])
    b, f = {"fp": (4 * (nvox + nproj), 4 * samples),
            "bp": (4 * (nvox + nproj), 10 * updates),
            "filter": (8 * nproj, fft),
            # read x, b and both weights, write x and the residual
            "sart": (4 * (3 * nvox + 3 * nproj), 4 * samples + 10 * updates + 3 * (nvox + nproj)),
            # read x, xold, z, img and precon, write x and z
            "mom": (4 * 7 * nvox, 2 * MOM["steps"] * 20 * nvox),
            "fdk": (4 * (nvox + nproj), 4 * samples + 10 * updates + fft)}[case["kind"]]
    return {"bytes": float(b), "flops": float(f)}


# ------------------------------------------------------------------- exact
def _fp64(c, g, vol):
    """Ray-driven projection in 64 bits: n left-Riemann trilinear samples
    between the box faces, zero outside the volume."""
    n = int(np.float32(SPP) * np.float32(g.nx))
    f64 = dict(device=DEV, dtype=torch.float64)
    v5 = vol.double()[None, None]
    out = torch.empty(g.proj_shape(c["views"]), **f64)
    u = ((torch.arange(g.nu, **f64) + 0.5) / g.nu - 0.5)[None, :] * g.fov_u
    v = ((torch.arange(g.nv, **f64) + 0.5) / g.nv - 0.5)[:, None] * g.fov_v
    half = (g.lx / 2, g.ly / 2, g.lz / 2)
    chunk = max(1, int(6e7 // (g.nu * g.nv)))
    for k, th in enumerate(_angles(c).astype(np.float64) * (math.pi / 180.0)):
        ct, st = math.cos(th), math.sin(th)
        src = (st * SAD, -ct * SAD, 0.0)
        d = [(ct * u - st * (SDD - SAD) - src[0]).expand(g.nv, g.nu),
             (st * u + ct * (SDD - SAD) - src[1]).expand(g.nv, g.nu), v.expand(g.nv, g.nu)]
        lo, hi = torch.zeros((g.nv, g.nu), **f64), torch.ones((g.nv, g.nu), **f64)
        for a in range(3):
            ta, tb = (half[a] - src[a]) / d[a], (-half[a] - src[a]) / d[a]
            lo, hi = torch.maximum(lo, torch.minimum(ta, tb)), torch.minimum(hi, torch.maximum(ta, tb))
        h = (hi - lo) / n
        # grid_sample's [-1, 1] is the box: its coordinates are 2 r / l
        p = torch.stack([(src[a] + lo * d[a]) / half[a] for a in range(3)], -1)
        q = torch.stack([d[a] * h / half[a] for a in range(3)], -1)
        acc = torch.zeros((g.nv, g.nu), **f64)
        for m0 in range(0, n, chunk):
            m = torch.arange(m0, min(n, m0 + chunk), **f64)[:, None, None, None]
            acc += torch.nn.functional.grid_sample(v5, (p[None] + m * q[None])[None], mode="bilinear",
                                                   padding_mode="zeros", align_corners=False)[0, 0].sum(0)
        out[k] = acc * (torch.sqrt(d[0] ** 2 + d[1] ** 2 + d[2] ** 2) * h.abs())
    return out


def _bp64(c, g, proj, fbp):
    """Voxel-driven backprojection in 64 bits, bilinear, zero outside."""
    f64 = dict(device=DEV, dtype=torch.float64)
    out = torch.zeros(g.vol_shape, **f64)
    x = (((torch.arange(g.nx, **f64) + 0.5) / g.nx - 0.5) * g.lx)[None, :]
    y = (((torch.arange(g.ny, **f64) + 0.5) / g.ny - 0.5) * g.ly)[:, None]
    z = (((torch.arange(g.nz, **f64) + 0.5) / g.nz - 0.5) * g.lz)[:, None, None]
    for k, th in enumerate(_angles(c).astype(np.float64) * (math.pi / 180.0)):
        ct, st = math.cos(th), math.sin(th)
        qx, qy = ct * x + st * y, ct * y - st * x
        mag = SDD / (qy + SAD)
        # box coordinates of the detector: 2 u / fov
        gu = (qx * mag * (2.0 / g.fov_u))[None].expand(g.nz, g.ny, g.nx)
        gv = z * (mag * (2.0 / g.fov_v))[None]
        s = torch.nn.functional.grid_sample(proj[k].double()[None, None], torch.stack([gu, gv], -1).reshape(1, g.nz, -1, 2),
                                            mode="bilinear", padding_mode="zeros", align_corners=False)
        s = s[0, 0].reshape(g.vol_shape)
        out += s / (((SAD - qy) / SAD) ** 2)[None] if fbp else s
    return out


def _parker64(c, g):
    """Short-scan weights (views, nu)."""
    f64 = dict(device=DEV, dtype=torch.float64)
    delta, eps = math.atan(g.fov_u / (2.0 * g.sdd)), 0.001
    beta = torch.from_numpy(_angles(c).astype(np.float64) * (math.pi / 180.0)).to(DEV)[:, None]
    alpha = -torch.atan((torch.arange(g.nu, **f64) / g.nu - 0.5) * 2.0 * math.tan(delta))[None, :]

    def S(b):
        return torch.where(b <= -0.5, 0.0, torch.where(b < 0.5, 0.5 * (1.0 + torch.sin(math.pi * b)), 1.0))

    def B(a):
        return 0.1 * (2.0 * (delta - a) + 0.001)

    return 0.5 * (S(beta / B(alpha) - 0.5) + S((beta + 2.0 * (alpha - delta) - eps) / B(alpha) + 0.5)
                  - S((beta - math.pi + 2.0 * alpha) / B(-alpha) - 0.5)
                  - S((beta - math.pi - 2.0 * delta - eps) / B(-alpha) + 0.5))


def _prefilter64(c, g, proj, F):
    """Cosine weights, short-scan weights, then the ramp filter: rows padded
    to 2 nu, times the response F[0..nu], cropped."""
    f64 = dict(device=DEV, dtype=torch.float64)
    u = ((torch.arange(g.nu, **f64) / g.nu - 0.5) * g.fov_u * (SAD / SDD))[None, :]
    v = ((torch.arange(g.nv, **f64) / g.nv - 0.5) * g.fov_v * (SAD / SDD))[:, None]
    w = SAD / torch.sqrt(SAD * SAD + u * u + v * v)
    parker = _parker64(c, g) if c.get("short") else None
    resp = torch.from_numpy(F.astype(np.float64)).to(DEV)
    out = torch.empty(proj.shape, **f64)
    step = max(1, int(3e7 // (g.nu * g.nv)))
    for k in range(0, c["views"], step):
        p = proj[k:k + step].double() * w
        if parker is not None:
            p = p * parker[k:k + step, None, :]
        out[k:k + step] = torch.fft.irfft(torch.fft.rfft(p, n=2 * g.nu) * resp, n=2 * g.nu)[..., :g.nu]
    return out


def _mom64(s):
    x, xold, z, img, P = (s[k].double() for k in ("x", "xold", "z", "img", "precon"))
    tl = MOM["tau"] / MOM["avg_lambda"]
    z = z + MOM["step"] * img * P
    for _ in range(MOM["steps"]):
        grad = [(torch.roll(x, -1, d) - x) * (MOM["weight"] * MOM["sigma"]) for d in (2, 1, 0)]
        den = torch.clamp(torch.sqrt(grad[0] ** 2 + grad[1] ** 2 + grad[2] ** 2), min=1.0)
        tv = torch.zeros_like(x)
        for q, d in zip(grad, (2, 1, 0)):
            q = q / den
            tv += torch.roll(q, 1, d) - q
        x = (x - MOM["tau"] * (tv * MOM["weight"]) + tl * z / P) / (1.0 + tl / P)
    x = torch.clamp(x, min=0.0)
    return {"x": x, "z": x * (1.0 + MOM["c"]) - MOM["c"] * xold}


def exact(case, seed):
    kind, g = case["kind"], _geom(case)
    samples = case["views"] * g.nu * g.nv * int(SPP * g.nx)
    updates = case["views"] * g.nx * g.ny * g.nz
    # about what 20 seconds allow
    if (kind in ("fp", "sart", "fdk") and samples > 1.2e10) or (kind in ("bp", "sart", "fdk") and updates > 1.2e10):
        return None
    s = _inputs(case, seed)
    if kind == "fp":
        return _fp64(case, g, s["vol"])
    if kind == "bp":
        return _bp64(case, g, s["proj"], case["fbp"])
    if kind == "filter":
        return _prefilter64(case, g, s["proj"], capi.default_filter(g.nu))
    if kind == "mom":
        return _mom64(s)
    if kind == "sart":
        r = (s["b"].double() - _fp64(case, g, s["x"])) * s["wp"].double()
        x = s["x"].double() + _bp64(case, g, r, False) * s["wx"].double()
        return {"x": torch.clamp(x, min=0.0), "r": r}
    # fdk: FBP, image *= 2 / views, then the least-squares scale of its projection
    q = _prefilter64(case, g, s["proj"], np.arange(g.nu + 1, dtype=np.float32))
    vol = _bp64(case, g, q, True) * (2.0 / case["views"])
    a, p = _fp64(case, g, vol), s["proj"].double()
    scale = float((a * p).sum() / (a * a).sum())
    return {"vol": vol * scale, "scale": np.float64(scale)}
