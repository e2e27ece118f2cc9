"""What the fan-plane pair promises beyond its accuracy: forward and adjoint
hold the same matrix entry for entry, whichever columns a wavefront takes
together, the adjoint's fixed-point sums have no bias, and steep rays meet the
slices as exactly as level ones."""
import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"


def _matrices(vol, det, ang):
    """The projector's matrix [rays, voxels] from the forward (unit voxels) and
    from the adjoint (unit rays)."""
    import nefct_hip as nh
    nz, ny, nx = vol.shape_zyx
    voxels, rays = nz * ny * nx, ang.numel() * det.nb * det.na
    fwd = torch.empty((voxels, rays), device=DEV)
    adj = torch.empty((rays, voxels), device=DEV)
    x = torch.zeros(vol.shape_zyx, device=DEV)
    y = torch.zeros((ang.numel(), det.nb, det.na), device=DEV)
    for j in range(voxels):
        x.view(-1)[j] = 1.0
        fwd[j] = nh.project(x, vol, det, ang).reshape(-1)
        x.view(-1)[j] = 0.0
    for i in range(rays):
        y.view(-1)[i] = 1.0
        adj[i] = nh.backproject(y, vol, det, ang).reshape(-1)
        y.view(-1)[i] = 0.0
    return fwd.t().double(), adj.double()


@pytest.mark.parametrize("columns", ["one-slow-of-three", "fine"])
def test_forward_and_adjoint_hold_the_same_entries(columns):
    """Detector columns along a grid axis (whose rays find their own crossings)
    beside columns of other slopes in one group of four, and rays that leave the
    volume through its top and bottom: a column's entries are the same from
    either side.  An entry is a difference of slab fractions, each
    rounded to FP32 a few times on either side (6 * 2^-24 of a slab at most),
    times the millimetres per slab (sqrt(3) voxels at most)."""
    import nefct_hip as nh
    if columns == "fine":       # 0.011 rad between columns
        vol = nh.VolumeGeometry.cube((44, 40, 5), 1.0)
        det = nh.ConeGeometry.flat(120.0, 180.0, 30, 2.0, 5, 3.6)
    else:                       # slopes -1, 0 and 1 side by side
        vol = nh.VolumeGeometry.cube((36, 32, 6), 1.0)
        det = nh.ConeGeometry.flat(30.0, 60.0, 3, 58.0, 6, 3.0)
    ang = torch.tensor([0.004, math.pi / 2 + 0.007, math.pi - 0.011, -math.pi / 2 + 0.013])
    f, a = _matrices(vol, det, ang)
    assert int((f > 0).sum()) > 400
    off = (f - a).abs()
    assert float(off.max()) <= 6 * 2.0 ** -24 * math.sqrt(3.0), (float(off.max()), int((off > 1e-6).sum()))


def test_one_hot_projection_value_does_not_darken_the_image():
    """The fixed-point unit follows the largest projection value.  With one
    value 1e5 times the others (on a ray that misses the volume) a slab of the
    others is 2^30 / 1e5 = 1.07e4 units long at most; parts that are rounded to
    the nearest unit leave the image's mean within a tenth of a unit per slab."""
    import nefct_hip as nh
    vol = nh.VolumeGeometry.cube((48, 48, 48), 1.0)
    det = nh.ConeGeometry.flat(300.0, 450.0, 160, 1.3, 120, 1.3)
    ang = torch.linspace(0.2, 6.2, 40)
    y = torch.ones((40, det.nb, det.na), device=DEV)
    plain = nh.backproject(y, vol, det, ang).double()
    y[0, 0, 0] = 1e5
    alone = torch.zeros_like(y)
    alone[0, 0, 0] = 1.0
    assert not nh.backproject(alone, vol, det, ang).any()
    hot = nh.backproject(y, vol, det, ang).double()
    assert not torch.equal(hot, plain)
    bias = float((hot - plain).mean() / plain.mean())
    assert abs(bias) <= 0.1 * 1e5 * 2.0 ** -30, bias


def test_steep_rays_meet_the_slices_as_exactly_as_level_ones(oracle):
    """Slices of +-1 make a ray's sum a measure of where it crosses from slice
    to slice: every other crossing changes it by 2.  z on a ray
    is an FP32 number of at most 8 cells (the half height) plus a product of the
    same size: three roundings of 2^-22 cells at most, 1.4e-7 rms each, 2.4e-7
    together; steep rays (slope above 0.2) leave after half a dozen crossings:
    2.4e-7 * 2 * sqrt(6 / 2) = 8e-7 cells.  (An FP32 origin at the column's
    middle, where z reaches 60 cells, gave 1.4e-6.)"""
    import nefct_hip as nh
    vol = nh.VolumeGeometry.cube((256, 256, 16), 1.0)
    det = nh.ConeGeometry.flat(190.0, 300.0, 120, 5.0, 64, 6.0)
    ang = (0.37 + 2 * math.pi * np.arange(12) / 12).astype(np.float32)
    x = np.random.default_rng(0).choice([-1.0, 1.0], size=(16, 1, 1)) * np.ones(vol.shape_zyx)
    ov = oracle.vol_struct(vol.grid, vol.center, vol.size)
    od = oracle.det_struct(0, det.SID, det.SAD, det.na, det.da, det.ai, det.nb, det.db, det.bi)
    got = nh.project(torch.tensor(x, dtype=torch.float32, device=DEV), vol, det, torch.tensor(ang))
    off = got.double().cpu().numpy() - oracle.exact_fwd(ov, od, ang.astype(np.float64), x)
    inside = oracle.exact_fwd(ov, od, ang.astype(np.float64), np.ones(vol.shape_zyx)) > 0
    a = ((np.arange(det.na) + 0.5 - det.na / 2) * det.da)[None, None, :]
    b = np.abs((np.arange(det.nb) + 0.5 - det.nb / 2) * det.db)[None, :, None]
    slope = np.broadcast_to(b / np.sqrt(det.SAD ** 2 + a ** 2 + b ** 2), off.shape)
    steep = inside & (slope > 0.2)
    assert steep.sum() > 2000
    rms = float(np.sqrt(((off * slope)[steep] ** 2).mean()))
    assert rms <= 8e-7, rms


@pytest.mark.parametrize("tilt", [0.0, 1e-7, 1e-5, 1e-3, 6e-3])
def test_constant_volume_gives_the_chord_on_slow_paths(tilt):
    """The middle column's ray through the volume's centre, along a cell face or
    crossing it slowly: its length is 48 / cos(tilt), whichever cells it is
    booked to.  At most 2 * 48 pieces added in FP32: 96 * 2^-24."""
    import nefct_hip as nh
    vol = nh.VolumeGeometry.cube((48, 48, 40), 1.0)
    det = nh.ConeGeometry.flat(300.0, 450.0, 65, 1.5, 70, 1.5)
    ang = torch.tensor([k * math.pi / 2 + s * tilt for k in range(4) for s in (1, -1)], dtype=torch.float32)
    ones = nh.project(torch.ones(vol.shape_zyx, device=DEV), vol, det, ang)[:, 35, 32].double()
    want = 48.0 / math.cos(tilt) * math.sqrt(1.0 + (0.75 / 450.0) ** 2)
    assert float((ones / want - 1.0).abs().max()) <= 96 * 2.0 ** -24
