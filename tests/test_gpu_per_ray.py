"""The exact pair where every ray is walked by itself: cones too steep for the
fan planes (rays that cross more than one slice per slab, some along z first),
with every block shape, lane spacing, forward tile and summing variant, split
and unsplit views and batches; and detectors of few rows, whose forward and
adjoint may each take another walk.  Every geometry is asserted to walk as its
test means.  Tolerances are the pair's own: 1e-5 against the FP64 oracle, 1e-6
for the transpose."""
import ctypes
import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"


def _steep():
    import nefct_hip as nh
    from nefct_hip.autotune import walks_fan_planes
    vol = nh.VolumeGeometry((70, 45, 37), (2.0, -3.0, 1.0), (70.0, 45.0, 37 * 1.2))
    det = nh.ConeGeometry.flat(60.0, 90.0, 90, 1.6, 70, 2.4, ai=0.2, bi=0.4)
    ang = np.concatenate([np.float32(math.pi / 4) + np.float32(0.004) * np.arange(-3, 4),
                          2 * math.pi * np.arange(9) / 9 + 0.1]).astype(np.float32)
    for adjoint in (False, True):
        assert not walks_fan_planes(vol, det, ang.size, 0, adjoint)
    return vol, det, ang


def _sino(det, ang, signed):
    rng = np.random.default_rng(23 + int(signed))
    return (rng.standard_normal if signed else rng.uniform)(size=(ang.size, det.nb, det.na)).astype(np.float32)


def _oracle_geometry(oracle, vol, det):
    return (oracle.vol_struct(vol.grid, vol.center, vol.size),
            oracle.det_struct(det.cyl, det.SID, det.SAD, det.na, det.da, det.ai, det.nb, det.db, det.bi))


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def _adjoint_into_nan(y, vol, det, ang, flags, entry="nefct_backproject_flat"):
    from nefct_hip import _lib, ops
    nx, ny, nz = vol.grid
    out = torch.full((nz, ny, nx), float("nan"), device=DEV)
    a = ang.to(DEV)
    ws, nbytes = ops._workspace(list(vol.grid), a.numel(), y.device)
    room = () if entry.endswith("noalloc") else (ops._ptr(ws), nbytes)
    st = getattr(_lib.load(), entry)(
        ops._ptr(y), _lib.int3(vol.grid), _lib.float3(vol.center), _lib.float3(vol.size), ops._ptr(a), a.numel(),
        det.SID, det.SAD, det.na, det.da, det.ai, det.nb, det.db, det.bi, ops._ptr(out), int(flags), *room,
        ctypes.c_void_p(ops._stream_ptr(y.device)))
    _lib.check(st, entry)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("signed", [False, True])
def test_steep_adjoint_bitwise_across_shapes_and_splits(oracle, signed):
    from nefct_hip import _lib as L
    vol, det, ang = _steep()
    yn = _sino(det, ang, signed)
    y, a = torch.tensor(yn, device=DEV), torch.tensor(ang)
    # 18 blocks: the default splits the views, the allocation-free call cannot
    base = _adjoint_into_nan(y, vol, det, a, 0, "nefct_backproject_flat_noalloc")
    assert torch.isfinite(base).all()
    for shape in (L.F_TILE_32x32x16, L.F_TILE_64x32x8, L.F_TILE_64x16x16, L.F_TILE_32x32x8, L.F_TILE_32x16x8,
                  L.F_TILE_16x16x32):
        for stride in (0, L.F_LANE_STRIDE2):
            got = _adjoint_into_nan(y, vol, det, a, shape | stride)
            assert torch.equal(got.view(torch.int32), base.view(torch.int32)), hex(shape | stride)
    ov, od = _oracle_geometry(oracle, vol, det)
    ref = oracle.exact_bp(ov, od, ang.astype(np.float64), yn.astype(np.float64))
    assert _rel(base.double().cpu().numpy(), ref) < 1e-5


@pytest.mark.parametrize("variant", ["float", "float64x32x8", "window", "ordered"])
def test_steep_summing_variants(oracle, variant):
    import nefct_hip as nh
    from nefct_hip import _lib as L
    vol, det, ang = _steep()
    flags = {"float": L.F_ADJ_FLOAT_ATOMIC, "float64x32x8": L.F_ADJ_FLOAT_ATOMIC | L.F_TILE_64x32x8,
             "window": L.F_ADJ_WINDOW, "ordered": L.F_ADJ_FLOAT_ATOMIC | L.F_DETERMINISTIC}[variant]
    ov, od = _oracle_geometry(oracle, vol, det)
    for signed in (False, True):
        yn = _sino(det, ang, signed)
        y = torch.tensor(yn, device=DEV)
        got = nh.backproject(y, vol, det, torch.tensor(ang), flags=flags)
        ref = oracle.exact_bp(ov, od, ang.astype(np.float64), yn.astype(np.float64))
        assert _rel(got.double().cpu().numpy(), ref) < 1e-5
        if variant == "ordered":
            assert torch.equal(got, nh.backproject(y, vol, det, torch.tensor(ang), flags=flags))


def test_steep_forward_tiles_and_transpose(oracle):
    import nefct_hip as nh
    from nefct_hip import _lib as L
    vol, det, ang = _steep()
    a = torch.tensor(ang)
    x = torch.randn(vol.shape_zyx, generator=torch.Generator().manual_seed(1))
    p = nh.project(x.to(DEV), vol, det, a)
    for tile in (L.F_FWD_TILE_32x8, L.F_FWD_TILE_8x32, L.F_FWD_TILE_64x4):
        assert torch.equal(nh.project(x.to(DEV), vol, det, a, flags=tile | L.fwd_vg(3)), p), hex(tile)
    ov, od = _oracle_geometry(oracle, vol, det)
    ref = oracle.exact_fwd(ov, od, ang.astype(np.float64), x.double().numpy())
    assert _rel(p.double().cpu().numpy(), ref) < 1e-5
    y = torch.tensor(_sino(det, ang, True), device=DEV)
    lhs = float((p.double() * y.double()).sum())
    rhs = float((x.to(DEV).double() * nh.backproject(y, vol, det, a).double()).sum())
    assert abs(lhs - rhs) <= 1e-6 * float((p.double() * y.double()).abs().sum())


@pytest.mark.parametrize("signed", [False, True])
def test_steep_batch_equals_plain_for_both_lane_spacings(signed):
    import nefct_hip as nh
    from nefct_hip import _lib as L
    from nefct_hip.batch import SiddonBatch
    vol, det, ang = _steep()
    small = (nh.VolumeGeometry.cube((24, 24, 24), 1.0), nh.ConeGeometry.flat(30.0, 45.0, 12, 4.0, 40, 6.0), ang[:6])
    b = SiddonBatch([(vol, det, ang), small])
    assert [p.pad_ for p in b.host] == [0, 0]
    ys = [torch.tensor(_sino(d, a, signed), device=DEV) for _, d, a in ((vol, det, ang), small)]
    for flags in (0, L.F_LANE_STRIDE2):
        for s, y in zip(b.sinograms, ys):
            s.copy_(y)
        b.flags = flags
        b.backproject()
        for v, y, (vo, d, a) in zip(b.volumes, ys, ((vol, det, ang), small)):
            assert torch.equal(v, nh.backproject(y, vo, d, torch.tensor(a)))


# (volume, columns, rows, views, row pitch): forward and adjoint on fan planes or not
@pytest.mark.parametrize("grid, na, nb, nv, db, forward, adjoint", [
    ((160, 150, 12), 320, 12, 120, 1.5, False, True),       # few rows, few blocks
    ((330, 330, 4), 500, 4, 40, 1.5, False, False),         # few rows, many blocks
    ((120, 130, 90), 240, 45, 60, 3.1, False, True),        # rows two voxels apart
    ((64, 64, 1), 128, 1, 12, 1.5, True, False),            # one row, hardly any work
])
def test_few_or_distant_rows(oracle, grid, na, nb, nv, db, forward, adjoint):
    """A forward per ray and an adjoint on fan planes are transposes up to
    rounding, too."""
    import nefct_hip as nh
    from nefct_hip.autotune import walks_fan_planes
    vol = nh.VolumeGeometry.cube(grid, 1.0)
    # (bi a little off the middle: no ray in the face between two slices)
    det = nh.ConeGeometry.flat(1000.0, 1500.0, na, max(grid[:2]) * 1.5 / na, nb, db, bi=0.55)
    ang = (0.2 + 2 * math.pi * np.arange(nv) / nv).astype(np.float32)
    assert walks_fan_planes(vol, det, nv, 0, False) == forward
    assert walks_fan_planes(vol, det, nv, 0, True) == adjoint
    rng = np.random.default_rng(8)
    x = rng.uniform(0, 1, vol.shape_zyx).astype(np.float32)
    y = rng.uniform(0, 1, (nv, nb, na)).astype(np.float32)
    p = nh.project(torch.tensor(x, device=DEV), vol, det, torch.tensor(ang)).double().cpu().numpy()
    b = nh.backproject(torch.tensor(y, device=DEV), vol, det, torch.tensor(ang)).double().cpu().numpy()
    ov, od = _oracle_geometry(oracle, vol, det)
    assert _rel(p, oracle.exact_fwd(ov, od, ang.astype(np.float64), x.astype(np.float64))) < 1e-5
    assert _rel(b, oracle.exact_bp(ov, od, ang.astype(np.float64), y.astype(np.float64))) < 1e-5
    lhs, rhs = float((p * y).sum()), float((b * x).sum())
    assert abs(lhs - rhs) <= 1e-6 * abs(lhs)
