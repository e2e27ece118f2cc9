"""The work a user of this package has it do, as cases that can be timed.

Every case is one call (or one forward + backward) through a public entry
point of ``nefct_hip``: the projector pair on its own, under autograd, in the
reference's op form, batched and behind a warp, FDK, a descent with total
variation and the inverse warp.  Sizes are the package's own workloads (C1, C2,
C4, C5 of nefct_hip/configs.py, the smoke test's volume) and odd sizes between
them.  Inputs are made on the device from the seed alone: ellipsoid phantoms,
their analytic line integrals with Poisson-like noise, smooth displacement
fields.
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "ct-nef_amd"))

import nefct_hip as nh  # noqa: E402
from nefct_hip import deform as nh_deform  # noqa: E402
from nefct_hip import fdk as nh_fdk  # noqa: E402
from nefct_hip import recon as nh_recon  # noqa: E402
from nefct_hip import reference as nh_ref  # noqa: E402
from nefct_hip.batch import SiddonBatch, batched_project  # noqa: E402
from nefct_hip.fourd import warp_project  # noqa: E402

DEV = "cuda"


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------
def _scan(name, kind, grid, voxel, na, nb, nv, sod=1000.0, sdd=1500.0, cyl=False, helical=False, **more):
    """A volume, a detector that covers it (pitch = extent * sdd / sod / cells,
    an angle on a cylindrical detector) and a full circle of nv views."""
    nx, ny, nz = grid
    case = {"name": name, "kind": kind, "nx": nx, "ny": ny, "nz": nz, "voxel": voxel, "na": na, "nb": nb, "nv": nv,
            "sod": sod, "sdd": sdd, "da": max(nx, ny) * voxel * sdd / sod / na / (sdd if cyl else 1.0),
            "db": nz * voxel * sdd / sod / nb, "cyl": cyl, "helical": helical}
    case.update(more)
    return case


def listed():
    return [
        # a unit-test sized projection: the call's fixed cost, launches and host path
        _scan("project_tiny", "project", (32, 32, 32), 4.0, 64, 48, 12, da=6.0, db=6.0),
        # backprojection of the smallest volume of the uneven batch: few voxels, many views
        _scan("backproject_64", "backproject", (64, 64, 64), 1.0, 128, 128, 120, sod=700.0, sdd=1050.0),
        # the C1 workload under autograd: A x, and A^T of the residual
        _scan("pair_c1", "pair", (128, 128, 128), 1.0, 256, 256, 180, da=1.5, db=1.5),
        # the C2 workload, the package's headline size: all 720 views forward ...
        _scan("project_c2", "project", (512, 512, 256), 0.8, 1024, 768, 720, da=0.6, db=0.6),
        # ... and back
        _scan("backproject_c2", "backproject", (512, 512, 256), 0.8, 1024, 768, 720, da=0.6, db=0.6),
        # a helical scan on a cylindrical detector, no size a multiple of anything
        _scan("helical_cyl", "both", (201, 187, 90), 1.1, 333, 117, 97, sod=570.0, sdd=1040.0, cyl=True,
              helical=True),
        # the reference's own ops ProjectFlat / BackProjectFlat, with its arithmetic
        _scan("reference_ops", "reference", (128, 128, 128), 1.0, 256, 256, 90, da=1.5, db=1.5),
        # uneven problems (sides of the C5 workload) batched, forward and backward
        _scan("batch_uneven", "batch", (128, 128, 128), 1.0, 256, 256, 0, problems=8),
        # 4-D CT (C4): ten warped phases of one volume, gradients to volume and displacement fields
        _scan("warp_project_c4", "warp_project", (256, 256, 160), 1.0, 384, 288, 0, problems=10),
        # FDK of the C2 short scan with Parker weights
        _scan("fdk_c2_short", "fdk", (512, 512, 256), 0.8, 1024, 768, 408, da=0.6, db=0.6, parker=True,
              window="ram-lak"),
        # an iterative reconstruction: descent steps on 0.5 |A x - b|^2 + lam TV(x)
        _scan("descent_c1", "descent", (128, 128, 128), 1.0, 256, 256, 180, da=1.5, db=1.5, steps=6),
        # motion compensation: warp by the inverse of a displacement field
        {"name": "deform_invert", "kind": "deform_invert", "nx": 256, "ny": 256, "nz": 160, "voxel": 1.0},
    ]


def draw(rng):
    """One more case: any of the kinds, sides 32 to 288, detectors of 0.7 to
    2.2 cells per voxel of the side, 12 to 400 views, flat or cylindrical."""
    kind = rng.choice(["project", "backproject", "pair", "both", "reference", "batch", "warp_project", "fdk",
                       "descent", "deform_invert"])

    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    big = {"batch": 144, "warp_project": 224, "descent": 144, "reference": 192}.get(kind, 288)
    nx = log(32, big)
    ny = nx if rng.random() < 0.5 else min(big, max(24, int(nx * rng.uniform(0.75, 1.3))))
    nz = min(big, max(8, int(nx * rng.uniform(0.3, 1.1))))
    voxel = round(rng.uniform(0.5, 2.0), 3)
    if kind == "deform_invert":
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "voxel": voxel}
    na = int(max(nx, ny) * rng.uniform(0.7, 2.2))
    nb = max(4, int(nz * rng.uniform(0.7, 2.2)))
    nv = log(12, 400)
    half = 0.75 * max(nx, ny) * voxel
    sod = round(half * rng.uniform(2.5, 8.0), 2)
    sdd = round(sod * rng.uniform(1.3, 1.8), 2)
    single = kind in ("project", "backproject", "both", "pair")
    case = _scan("", kind, (nx, ny, nz), voxel, na, nb, nv, sod=sod, sdd=sdd, cyl=single and rng.random() < 0.3,
                 helical=single and kind != "pair" and rng.random() < 0.3)
    del case["name"]
    if kind == "reference":
        case["db"] = case["da"]     # the op knows one pitch
    if kind in ("batch", "warp_project"):
        case["problems"] = rng.randint(2, 8)
        case["nv"] = 0
    if kind == "fdk":
        case["parker"] = rng.random() < 0.4
        case["window"] = rng.choice(["ram-lak", "shepp-logan", "hann", "hamming", "cosine"])
    if kind == "descent":
        case["steps"] = rng.randint(2, 6)
    return case


# --------------------------------------------------------------------------
# geometry and inputs
# --------------------------------------------------------------------------
def _geometry(case):
    v = case["voxel"]
    vol = nh.VolumeGeometry.cube((case["nx"], case["ny"], case["nz"]), v)
    if case["cyl"]:
        det = nh.ConeGeometry("cyli", case["sod"], case["sdd"], case["na"], case["da"], 0.5, case["nb"], case["db"],
                              0.5)
    else:
        det = nh.ConeGeometry.flat(case["sod"], case["sdd"], case["na"], case["da"], case["nb"], case["db"])
    return vol, det


def _angles(case, rng):
    nv = case["nv"]
    step = 2 * math.pi / nv
    if case["kind"] == "fdk" and case["parker"]:     # a short scan: half a turn and the fan
        step = (math.pi + 2 * math.atan(case["na"] * case["da"] / 2 / case["sdd"])) / nv
    return (rng.uniform(0, 1) + step * np.arange(nv)).astype(np.float32)


def _offsets(case):
    """A helical scan's lift of source and detector per view (mm): a fifth of
    the volume's height over the scan (no view at zero lift, where a detector's
    middle row would lie in the face between two slices and belong to neither)."""
    if not case["helical"]:
        return None
    h = case["nz"] * case["voxel"]
    return np.linspace(-0.11 * h, 0.0917 * h, case["nv"]).astype(np.float32)


def _ellipsoids(vol, rng, count):
    """(centre, M, mu): the ellipsoid |M (p - centre)| <= 1; semi-axes 4 % to
    40 % of half the volume's sides."""
    out = []
    half = 0.5 * np.asarray(vol.size)
    for _ in range(count):
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        axes = rng.uniform(0.04, 0.4, 3) * half.min()
        out.append((rng.uniform(-0.55, 0.55, 3) * half, (q.T / axes[:, None]), rng.uniform(0.01, 0.03)))
    return out


def _phantom(vol, ells):
    nx, ny, nz = vol.grid
    ax = [torch.arange(n, device=DEV, dtype=torch.float32).add_(0.5).mul_(vs).sub_(s / 2)
          for n, vs, s in zip(vol.grid, vol.voxel, vol.size)]
    img = torch.zeros((nz, ny, nx), device=DEV)
    for c, M, mu in ells:
        r2 = 0
        for row in M:
            u = ((ax[0] - c[0]) * row[0])[None, None, :] + ((ax[1] - c[1]) * row[1])[None, :, None] \
                + ((ax[2] - c[2]) * row[2])[:, None, None]
            r2 = r2 + u * u
        img += (r2 <= 1) * float(mu)
    return img


def _line_integrals(det, ang, off, ells):
    """The phantom's analytic sinogram [nv, nb, na] (FP32)."""
    nv = len(ang)
    out = torch.zeros((nv, det.nb, det.na), device=DEV)
    u = (torch.arange(det.na, device=DEV, dtype=torch.float32) + det.ai) * det.da - det.na * det.da / 2
    v = (torch.arange(det.nb, device=DEV, dtype=torch.float32) + det.bi) * det.db - det.nb * det.db / 2
    lx = det.SAD * torch.cos(u) if det.cyl else torch.full_like(u, det.SAD)     # from the source
    ly = det.SAD * torch.sin(u) if det.cyl else u
    per = max(1, 16_000_000 // (det.na * det.nb))
    for v0 in range(0, nv, per):
        a = torch.tensor(np.asarray(ang[v0:v0 + per], np.float64), device=DEV)
        c, s = torch.cos(a).float()[:, None], torch.sin(a).float()[:, None]
        dx, dy = lx * c - ly * s, lx * s + ly * c                              # [views, na]
        z0 = torch.zeros_like(c) if off is None else torch.tensor(off[v0:v0 + per], device=DEV)[:, None]
        length = torch.sqrt(dx * dx + dy * dy)[:, None, :] ** 2 + (v * v)[None, :, None]
        length = torch.sqrt(length)
        for cen, M, mu in ells:
            A = B = 0
            C = -1.0
            for row in M:
                w = ((-det.SID * c - cen[0]) * row[0] + (-det.SID * s - cen[1]) * row[1] + (z0 - cen[2]) * row[2])
                d = (dx * row[0] + dy * row[1])[:, None, :] + (v * row[2])[None, :, None]
                A = A + d * d
                B = B + d * w[:, :, None]
                C = C + (w * w)[:, :, None]
            out[v0:v0 + per] += (2 * float(mu)) * torch.sqrt((B * B - A * C).clamp_min_(0)) / A * length
    return out


def _noisy(p, seed):
    """Transmission noise of 1e5 photons on line integrals."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    n = torch.randn(p.shape, generator=g, device=DEV)
    return p.add_(n.mul_(torch.exp(0.5 * p).mul_(1e5 ** -0.5)))


def _noise(shape, seed, scale):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(shape, generator=g, device=DEV) * scale


def _dvf(shape, rng, voxel):
    """Displacement field [3, nz, ny, nx] in voxels: Gaussian bumps, peak up to
    8 voxels along z and 3 across."""
    nz, ny, nx = shape
    i = [torch.arange(n, device=DEV, dtype=torch.float32) for n in (nx, ny, nz)]
    out = torch.zeros((3, nz, ny, nx), device=DEV)
    for _ in range(8):
        sg = rng.uniform(0.1, 0.25) * min(shape)
        c = rng.uniform(0, 1, 3) * (nx, ny, nz)
        e = [torch.exp(-(i[k] - c[k]) ** 2 / (2 * sg * sg)) for k in range(3)]
        b = e[2][:, None, None] * e[1][None, :, None] * e[0][None, None, :]
        for k, top in enumerate((3.0, 3.0, 8.0)):
            out[k] += b * float(min(top, 0.25 * sg) * rng.uniform(-1, 1))
    return out


def _problems(case, rng):
    """(volume, detector, angles) of a batched case."""
    out = []
    for p in range(case["problems"]):
        if case["kind"] == "warp_project":      # phases of one volume, their views scattered over the circle
            vol, det = _geometry(case)
            ang = np.sort(rng.uniform(0, 2 * math.pi, 40 + (23 * p + 40) % 81)).astype(np.float32)
        else:                                   # uneven cubes, (2 side)^2 detectors
            side = max(16, case["nx"] * (2, 3, 4, 6)[p % 4] // 4)
            sod = float(case["sod"] * (0.5 + 0.5 * ((p * 5) % 8) / 8))
            vol = nh.VolumeGeometry.cube((side, side, side), case["voxel"])
            pitch = case["voxel"] * 0.75
            det = nh.ConeGeometry.flat(sod, 1.5 * sod, 2 * side, pitch, 2 * side, pitch)
            nv = 60 + (37 * p) % 180
            ang = (2 * math.pi * np.arange(nv) / nv).astype(np.float32)
        out.append((vol, det, ang))
    return out


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "deform_invert":
        vol = nh.VolumeGeometry.cube((case["nx"], case["ny"], case["nz"]), case["voxel"])
        return {"kind": kind, "image": _phantom(vol, _ellipsoids(vol, rng, 12)),
                "dvf": _dvf(vol.shape_zyx, rng, case["voxel"])}
    if kind in ("batch", "warp_project"):
        probs = _problems(case, rng)
        st = {"kind": kind, "probs": probs, "batch": SiddonBatch(probs, device=DEV)}
        st["grads"] = [_noise((len(a), d.nb, d.na), seed + p, 0.02) for p, (_, d, a) in enumerate(probs)]
        if kind == "batch":
            st["volumes"] = [_phantom(v, _ellipsoids(v, rng, 8)).requires_grad_(True) for v, _, _ in probs]
        else:
            v = probs[0][0]
            st["base"] = _phantom(v, _ellipsoids(v, rng, 12)).requires_grad_(True)
            st["dvfs"] = [_dvf(v.shape_zyx, rng, case["voxel"]).requires_grad_(True) for _ in probs]
        return st
    vol, det = _geometry(case)
    ang, off = _angles(case, rng), _offsets(case)
    ells = _ellipsoids(vol, rng, 20)
    st = {"kind": kind, "vol": vol, "det": det, "ang": torch.tensor(ang, device=DEV),
          "off": None if off is None else torch.tensor(off, device=DEV)}
    if kind in ("project", "both", "reference", "pair"):
        st["image"] = _phantom(vol, ells).requires_grad_(kind == "pair")
    if kind in ("backproject", "both", "fdk", "descent", "reference"):
        st["sino"] = _noisy(_line_integrals(det, ang, off, ells), seed + 1)
    if kind == "pair":     # the residual of a fit: signed, noise-like
        st["grad"] = _noise((case["nv"], det.nb, det.na), seed + 2, 0.02)
    if kind == "fdk":
        st.update(host_angles=ang, parker=case["parker"], window=case["window"])
    if kind == "descent":
        st.update(steps=case["steps"], lipschitz=_lipschitz(case))
    return st


def _lipschitz(case):
    """Bound on |A^T A|: longest chord times the most a voxel collects."""
    v, mag = case["voxel"], case["sdd"] / case["sod"]
    chord = v * math.sqrt(case["nx"] ** 2 + case["ny"] ** 2 + case["nz"] ** 2)
    return 1.3 * chord * case["nv"] * v ** 3 * mag ** 2 / (case["da"] * case["db"])


LAM, EPS = 1e-3, 1e-6


def run(state):
    s, kind = state, state["kind"]
    if kind == "deform_invert":
        d = s["dvf"]
        return nh_deform.deform_invert_tex(s["image"], d[0], d[1], d[2])
    if kind == "batch":
        outs = batched_project(s["batch"], s["volumes"])
        grads = torch.autograd.grad(outs, s["volumes"], s["grads"])
        return [o.detach() for o in outs], list(grads)
    if kind == "warp_project":
        n = len(s["dvfs"])
        outs = warp_project(s["batch"], [s["base"]] * n, s["dvfs"])
        grads = torch.autograd.grad(outs, [s["base"]] + s["dvfs"], s["grads"])
        return [o.detach() for o in outs], list(grads)
    vol, det, ang, off = s["vol"], s["det"], s["ang"], s["off"]
    if kind == "project":
        return nh.project(s["image"], vol, det, ang, offsets=off)
    if kind == "backproject":
        return nh.backproject(s["sino"], vol, det, ang, offsets=off)
    if kind == "both":
        return nh.project(s["image"], vol, det, ang, offsets=off), nh.backproject(s["sino"], vol, det, ang, offsets=off)
    if kind == "pair":
        y = nh.forward_project(s["image"], vol, det, ang)
        (g,) = torch.autograd.grad(y, [s["image"]], [s["grad"]])
        return y.detach(), g
    if kind == "reference":
        args = (vol.grid, vol.center, vol.size, ang, det.SID, det.SAD, det.na, det.da, det.ai, det.nb, det.db, det.bi)
        return nh_ref.ProjectFlat(s["image"], *args), nh_ref.BackProjectFlat(s["sino"], *args, *vol.grid)
    if kind == "fdk":
        return nh_fdk.fdk(s["sino"], vol, det, s["host_angles"], parker=s["parker"], window=s["window"])
    if kind == "descent":
        x, history = nh_recon.gradient_descent(s["sino"], vol, det, ang, steps=s["steps"], lam=LAM, eps=EPS,
                                               lipschitz=s["lipschitz"])
        return x, history
    raise ValueError(kind)


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def _pair_work(nx, ny, nz, na, nb, nv):
    """Bytes and flops of one direction: volume and sinogram once; a multiply
    and an add per voxel a ray meets (a ray through the volume's middle meets
    about 0.9 side, and the detector's rim sees less)."""
    return 4.0 * (nx * ny * nz + na * nb * nv), 2.0 * na * nb * nv * 0.85 * 0.5 * (nx + ny)


def work(case):
    kind = case["kind"]
    vox = float(case["nx"]) * case["ny"] * case["nz"]
    if kind == "deform_invert":
        # 30 iterations of three trilinear samples (about 24 flops each), then the warp
        return {"bytes": 4.0 * vox * 5, "flops": vox * 24.0 * 91}
    if kind in ("batch", "warp_project"):
        b = f = 0.0
        for vol, det, ang in _problems(case, np.random.default_rng(0)):
            wb, wf = _pair_work(*vol.grid, det.na, det.nb, len(ang))
            n = float(np.prod(vol.grid))
            b, f = b + 2 * wb, f + 2 * wf
            if kind == "warp_project":      # the field in, its gradient out, the two warps' arithmetic
                b, f = b + 4.0 * n * 6, f + 100.0 * n
        return {"bytes": b, "flops": f}
    wb, wf = _pair_work(case["nx"], case["ny"], case["nz"], case["na"], case["nb"], case["nv"])
    if kind == "fdk":
        rays = float(case["na"]) * case["nb"] * case["nv"]
        # 14 flops per voxel and view; the filter's two FFTs over padded rows
        return {"bytes": wb, "flops": 14.0 * vox * case["nv"] + rays * 10.0 * math.log2(4 * case["na"])}
    times = {"project": 1, "backproject": 1, "pair": 2, "both": 2, "reference": 2,
             "descent": 2 * case.get("steps", 0)}[kind]
    return {"bytes": wb * times, "flops": wf * times}


# --------------------------------------------------------------------------
# 64-bit values, in plain torch
# --------------------------------------------------------------------------
def _f32(v):
    """A parameter as the entry points take it (rounded to FP32)."""
    return float(np.float32(v))


class _Walk64:
    """Every (ray, voxel, length) of a scan in FP64: per ray the axis of its
    largest step in voxels, one slab of that axis at a time, at most three
    voxels per slab.  ``rule``: None (exact lengths), "fwd" or "adj" (the
    reference op's attribution of a slab's pieces, 1/L^2 scale and short-ray
    skip)."""

    def __init__(self, vol, det, ang, off=None, rule=None):
        self.n, self.rule, self.det = vol.grid, rule, det
        self.vs = [_f32(s) / n for s, n in zip(vol.size, vol.grid)]
        self.lo = [_f32(c) - _f32(s) * 0.5 for c, s in zip(vol.center, vol.size)]
        self.ang = torch.as_tensor(ang).to(DEV).double()
        self.off = torch.zeros_like(self.ang) if off is None else torch.as_tensor(off).to(DEV).double()

    def _chunk(self, v0, v1):
        det, kw = self.det, dict(device=DEV, dtype=torch.float64)
        sid, sad = _f32(det.SID), _f32(det.SAD)
        a = (torch.arange(det.na, **kw) + _f32(det.ai)) * _f32(det.da) - det.na * _f32(det.da) / 2
        b = (torch.arange(det.nb, **kw) + _f32(det.bi)) * _f32(det.db) - det.nb * _f32(det.db) / 2
        lx = sad * torch.cos(a) - sid if det.cyl else torch.full_like(a, sad - sid)
        ly = sad * torch.sin(a) if det.cyl else a
        c, s = torch.cos(self.ang[v0:v1])[:, None, None], torch.sin(self.ang[v0:v1])[:, None, None]
        dz = self.off[v0:v1][:, None, None]
        S = [-sid * c, -sid * s, dz]
        D = [lx * c - ly * s, lx * s + ly * c, b[None, :, None] + dz]
        shape = (v1 - v0, det.nb, det.na)
        S = [x.expand(shape).reshape(-1) for x in S]
        return S, [x.expand(shape).reshape(-1) for x in D]

    def pieces(self, v0, v1):
        """Yields (index, weight, scale) per slab and piece of the rays of views v0..v1."""
        S, D = self._chunk(v0, v1)
        d = [(D[i] - S[i]) / self.vs[i] for i in range(3)]
        u = [(S[i] - self.lo[i]) / self.vs[i] for i in range(3)]
        live = torch.ones_like(d[0], dtype=torch.bool)
        if self.rule:
            xd, yd, zd = [(D[i] - S[i]) / self.vs[0] for i in range(3)]
            isx = (xd.abs() > yd.abs()) if self.rule == "adj" else (xd.abs() >= yd.abs())
            isz = torch.zeros_like(isx)
            if self.rule == "adj":
                live = torch.sqrt(xd * xd + yd * yd) >= 10
        else:
            ax, ay, az = [x.abs() for x in d]
            isx = (ax >= ay) & (ax >= az)
            isz = ~isx & (ay < az)
        nx, ny, nz = self.n

        def sel(x, y, z):      # the value for walk axis x, y or z
            x, y, z = [torch.as_tensor(q, device=DEV, dtype=torch.float64) for q in (x, y, z)]
            return torch.where(isx, x, torch.where(isz, z, y))

        dm, um, nm, vm = sel(*d), sel(*u), sel(*self.n), sel(*self.vs)
        ka, kb = sel(d[1], d[0], d[0]) / dm, sel(d[2], d[2], d[1]) / dm
        A, B = sel(u[1], u[0], u[0]) - ka * um, sel(u[2], u[2], u[1]) - kb * um
        na, nb = sel(ny, nx, nx), sel(nz, nz, ny)
        st_m, st_a, st_b = sel(1, nx, nx * ny), sel(nx, 1, 1), sel(nx * ny, nx * ny, nx)
        qa, qb = ka * sel(self.vs[1], self.vs[0], self.vs[0]) / vm, kb * sel(self.vs[2], self.vs[2], self.vs[1]) / vm
        scale = vm * torch.sqrt(1 + qa * qa + qb * qb)
        if self.rule == "fwd":
            scale = scale / (xd * xd + yd * yd + zd * zd)
        inva = torch.where(ka != 0, 1 / ka, torch.zeros_like(ka))
        invb = torch.where(kb != 0, 1 / kb, torch.zeros_like(kb))
        one = torch.ones_like(ka)
        # pieces outside the volume add nothing, each to a voxel of its own
        # (one voxel for all of them would serialise the adjoint's additions)
        spare = torch.arange(ka.numel(), device=DEV) % (nx * ny * nz)
        for t in range(max(self.n)):
            a0, b0 = A + ka * t, B + kb * t
            a1, b1 = A + ka * (t + 1), B + kb * (t + 1)
            ca0, ca1, cb0, cb1 = a0.floor(), a1.floor(), b0.floor(), b1.floor()
            ok = live & (t < nm)
            if self.rule:
                la, ha, lb, hb = (torch.minimum(ca0, ca1), torch.maximum(ca0, ca1), torch.minimum(cb0, cb1),
                                  torch.maximum(cb0, cb1))
                fa = torch.where(la != ha, (ha - torch.minimum(a0, a1)) * inva.abs(), one)
                fb = torch.where(lb != hb, (hb - torch.minimum(b0, b1)) * invb.abs(), one)
                ok = ok & (la >= torch.where(la == ha, 0.0, -1.0)) & (la < na)
                ok = ok & (lb >= torch.where(lb == hb, 0.0, -1.0)) & (lb < nb)
                ca0, ca1, cb0, cb1 = la, ha, lb, hb
                first = ~(fa > fb)
            else:
                fa = torch.where(ca1 != ca0, ((ca0 + (ka > 0).double() - a0) * inva).clamp(0, 1), one)
                fb = torch.where(cb1 != cb0, ((cb0 + (kb > 0).double() - b0) * invb).clamp(0, 1), one)
                first = fa < fb
            f1, f2 = torch.minimum(fa, fb), torch.maximum(fa, fb)
            for ca, cb, w in ((ca0, cb0, f1), (torch.where(first, ca1, ca0), torch.where(first, cb0, cb1), f2 - f1),
                              (ca1, cb1, 1 - f2)):
                keep = ok & (ca >= 0) & (ca < na) & (cb >= 0) & (cb < nb)
                idx = (t * st_m + ca * st_a + cb * st_b).long()
                yield torch.where(keep, idx, spare), torch.where(keep, w, 0.0), scale

    def _chunks(self):
        per = max(1, 3_000_000 // (self.det.na * self.det.nb))
        nv = self.ang.numel()
        return [(v, min(nv, v + per)) for v in range(0, nv, per)]

    def forward(self, image):
        img = image.detach().double().reshape(-1)
        out = torch.empty((self.ang.numel(), self.det.nb, self.det.na), dtype=torch.float64, device=DEV)
        for v0, v1 in self._chunks():
            acc = 0
            for idx, w, scale in self.pieces(v0, v1):
                acc = acc + w * img[idx]
            out[v0:v1] = (acc * scale).reshape(out[v0:v1].shape)
        return out

    def adjoint(self, sino):
        nx, ny, nz = self.n
        out = torch.zeros(nx * ny * nz, dtype=torch.float64, device=DEV)
        for v0, v1 in self._chunks():
            y = None
            for idx, w, scale in self.pieces(v0, v1):
                if y is None:
                    y = sino[v0:v1].detach().double().reshape(-1) * scale
                out.index_add_(0, idx, w * y)
        return out.reshape(nz, ny, nx)


def _warp64(image, dvf):
    """Trilinear warp with zero padding, differentiable, FP64.  The cell is
    the one the position rounded to FP32 lies in: at a voxel centre the
    interpolant has a kink, and its gradient there is that of either side."""
    nz, ny, nx = image.shape
    grid = torch.meshgrid(*[torch.arange(n, device=DEV, dtype=torch.float64) for n in image.shape], indexing="ij")
    p = [grid[2] + dvf[0], grid[1] + dvf[1], grid[0] + dvf[2]]
    base = [q.detach().float().floor().double() for q in p]
    f = [q - b for q, b in zip(p, base)]
    flat, out = image.reshape(-1), 0
    for corner in range(8):
        w, keep, i = 1, True, []
        for k, n in enumerate((nx, ny, nz)):
            up = (corner >> k) & 1
            w = w * (f[k] if up else 1 - f[k])
            q = base[k] + up
            keep = (q >= 0) & (q < n) & keep
            i.append(q.clamp(0, n - 1).long())
        out = out + torch.where(keep, w * flat[(i[2] * ny + i[1]) * nx + i[0]], 0.0)
    return out


def _clamped64(v, x, y, z):
    """Trilinear sample with edge texels repeated, at voxel coordinates."""
    nz, ny, nx = v.shape
    i, f = [], []
    for q, n in ((x, nx), (y, ny), (z, nz)):
        b = q.floor()
        f.append(q - b)
        i.append((b.clamp(0, n - 1).long(), (b + 1).clamp(0, n - 1).long()))
    flat, out = v.reshape(-1), 0
    for c in range(8):
        w = 1
        for k in range(3):
            w = w * (f[k] if (c >> k) & 1 else 1 - f[k])
        out = out + w * flat[(i[2][c >> 2] * ny + i[1][(c >> 1) & 1]) * nx + i[0][c & 1]]
    return out


def _ramp64(na, window):
    n = max(64, int(2 ** math.ceil(math.log2(2 * na))))
    k = np.arange(-(n // 2), n // 2)
    h = np.zeros(n)
    h[n // 2] = 0.25
    odd = k % 2 == 1
    h[odd] = -1.0 / (np.pi * k[odd]) ** 2
    half = (2 * np.abs(np.fft.fft(h)))[: n // 2 + 1]
    w = 2 * np.pi * np.arange(half.size) / n
    t = w[1:]
    half[1:] *= {"ram-lak": np.ones_like(t), "shepp-logan": np.sin(t / 2) / (t / 2), "cosine": np.cos(t / 2),
                 "hamming": 0.54 + 0.46 * np.cos(t), "hann": (1 + np.cos(t)) / 2}[window]
    return n, torch.tensor(half, device=DEV)


def _fdk64(sino, vol, det, ang, parker, window):
    kw = dict(device=DEV, dtype=torch.float64)
    nv, na, nb = len(ang), det.na, det.nb
    sid, sad, da, db = _f32(det.SID), _f32(det.SAD), _f32(det.da), _f32(det.db)
    ang = np.asarray(ang, np.float64)
    dang = abs(ang[1] - ang[0])
    dbeta = 2 * dang if parker else 2 * math.pi / nv
    scale = 1 / (2 * det.da) * dbeta / 2 * (det.SAD / det.SID)
    a = (torch.arange(na, **kw) + _f32(det.ai)) * da - na * da / 2
    b = (torch.arange(nb, **kw) + _f32(det.bi)) * db - nb * db / 2
    weight = sad * scale / torch.sqrt(sad * sad + (a * a)[None, :] + (b * b)[:, None])
    pk = torch.ones((nv, na), **kw)
    if parker:
        gam = torch.rad2deg(torch.atan(a / sad))
        fan = float((gam[-1] - gam[0]).abs()) / 2
        n180 = 180.0 / _f32(math.degrees(dang))
        pw = ((n180 - nv) / 2 + torch.arange(1, nv + 1, **kw)[:, None]) / n180 * 180.0 \
            + (1 if ang[1] > ang[0] else -1) * gam
        up = torch.sin(math.pi / 2 * (fan / 2 + pw) / fan).clamp_min(0) ** 2
        down = torch.cos(math.pi / 2 * (fan / 2 + pw - 180.0) / fan).clamp_min(0) ** 2
        pk = torch.where((pw <= fan / 2) & (pw > -fan / 2), up, pk)
        pk = torch.where((pw >= 180 - fan / 2) & (pw < 180 + fan / 2), down, pk)
        pk = torch.where((pw < -fan / 2) | (pw > 180 + fan / 2), 0.0, pk)
    n, resp = _ramp64(na, window)
    (nx, ny, nz), (vx, vy, vz) = vol.grid, [_f32(s) / q for s, q in zip(vol.size, vol.grid)]
    x = ((torch.arange(nx, **kw) + 0.5) * vx - _f32(vol.size[0]) / 2)[None, :]
    y = ((torch.arange(ny, **kw) + 0.5) * vy - _f32(vol.size[1]) / 2)[:, None]
    z = ((torch.arange(nz, **kw) + 0.5) * vz - _f32(vol.size[2]) / 2)[:, None, None]
    img = torch.zeros((nz, ny, nx), **kw)
    for iv in range(nv):
        q = sino[iv].double() * weight * pk[iv]
        q = torch.fft.irfft(torch.fft.rfft(q, n=n) * resp, n=n)[:, :na].contiguous().reshape(-1)
        c, s = math.cos(ang[iv]), math.sin(ang[iv])
        U = sid + x * c + y * s
        mag = sad / U
        fa = ((-x * s + y * c) * mag + na * da / 2) / da - _f32(det.ai)
        ia = fa.floor().clamp(0, max(na - 2, 0))
        ta = fa - ia
        w = torch.where((fa >= 0) & (fa <= na - 1), (sid / U) ** 2, 0.0)
        fb = z * (mag / db) + (nb * db / 2 / db - _f32(det.bi))
        ib = fb.floor().clamp(0, max(nb - 2, 0))
        tb = fb - ib
        j = (ib * na + ia).long()
        s0 = q[j] * (1 - ta) + q[j + 1] * ta
        s1 = q[j + na] * (1 - ta) + q[j + na + 1] * ta
        img += torch.where((fb >= 0) & (fb <= nb - 1), w * (s0 + tb * (s1 - s0)), 0.0)
    return img


def _tv64(x):
    """(sum sqrt(d^2 + eps^2), its gradient) over forward differences with a zero first slice."""
    value, grad = 0.0, torch.zeros_like(x)
    for k in range(3):
        d = torch.zeros_like(x)
        n = x.shape[k]
        d.narrow(k, 1, n - 1).copy_(x.narrow(k, 1, n - 1) - x.narrow(k, 0, n - 1))
        r = torch.sqrt(d * d + EPS * EPS)
        value += float(r.sum())
        ph = d / r
        grad += ph
        grad.narrow(k, 0, n - 1).sub_(ph.narrow(k, 1, n - 1))
    return value, grad


def exact(case, seed):
    kind = case["kind"]
    slabs = float(case.get("na", 0)) * case.get("nb", 0) * case.get("nv", 0) * max(case["nx"], case["ny"], case["nz"])
    if kind in ("project", "backproject", "pair", "both", "reference") and slabs > 1.2e10:
        return None
    if kind == "descent" and slabs * case["steps"] > 1.2e10:
        return None
    if kind == "fdk" and float(case["nx"]) * case["ny"] * case["nz"] * case["nv"] > 4e10:
        return None
    s = prepare(case, seed)
    with torch.no_grad():
        if kind == "deform_invert":
            m = s["dvf"].double()
            g = torch.meshgrid(*[torch.arange(n, device=DEV, dtype=torch.float64) for n in m.shape[1:]],
                               indexing="ij")
            d = [torch.zeros_like(g[0]) for _ in range(3)]
            for _ in range(30):
                for k in range(3):
                    d[k] = -_clamped64(m[k], g[2] + d[0], g[1] + d[1], g[0] + d[2])
            return _clamped64(s["image"].double(), g[2] + d[0], g[1] + d[1], g[0] + d[2])
        if kind in ("batch", "warp_project"):
            total = sum(float(d.na) * d.nb * len(a) * max(v.grid) for v, d, a in s["probs"])
            if total > 1.2e10:
                return None
            outs, grads = [], []
            for p, (vol, det, ang) in enumerate(s["probs"]):
                walk = _Walk64(vol, det, ang)
                if kind == "batch":
                    outs.append(walk.forward(s["volumes"][p]))
                    grads.append(walk.adjoint(s["grads"][p]))
                    continue
                gv = walk.adjoint(s["grads"][p])
                with torch.enable_grad():
                    base = s["base"].detach().double().requires_grad_(True)
                    dvf = s["dvfs"][p].detach().double().requires_grad_(True)
                    warped = _warp64(base, dvf)
                    gb, gd = torch.autograd.grad(warped, [base, dvf], gv)
                outs.append(walk.forward(warped))
                grads.append(gd)
                if p == 0:
                    total_base = gb
                else:
                    total_base = total_base + gb
            return (outs, grads) if kind == "batch" else (outs, [total_base] + grads)
        vol, det, ang, off = s["vol"], s["det"], s["ang"], s["off"]
        if kind == "reference":
            one = nh.ConeGeometry.flat(det.SID, det.SAD, det.na, det.da, det.nb, det.da)
            img = _Walk64(vol, det, ang, rule="adj").adjoint(s["sino"])
            return _Walk64(vol, one, ang, rule="fwd").forward(s["image"]), img.reshape(vol.grid)
        if kind == "fdk":
            return _fdk64(s["sino"], vol, det, s["host_angles"], s["parker"], s["window"])
        walk = _Walk64(vol, det, ang, off)
        if kind == "project":
            return walk.forward(s["image"])
        if kind == "backproject":
            return walk.adjoint(s["sino"])
        if kind == "both":
            return walk.forward(s["image"]), walk.adjoint(s["sino"])
        if kind == "pair":
            return walk.forward(s["image"]), walk.adjoint(s["grad"])
        x = torch.zeros(vol.shape_zyx, dtype=torch.float64, device=DEV)
        b, history = s["sino"].double(), []
        L = s["lipschitz"] * 1.05 + 12.0 * LAM / EPS
        for _ in range(s["steps"]):
            r = walk.forward(x) - b
            tv, g = _tv64(x)
            history.append(0.5 * float((r * r).sum()) + LAM * tv)
            x = x - (walk.adjoint(r) + LAM * g) / L
        return x, history


if __name__ == "__main__":
    for c in listed() + [draw(random.Random(i)) for i in range(4)]:
        print(c, work(c))
