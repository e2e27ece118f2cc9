"""What the fan-plane pair promises beyond its accuracy: forward and adjoint
hold the same matrix entry for entry, whichever columns a wavefront takes
together, and the adjoint's fixed-point sums have no bias."""
import math

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
