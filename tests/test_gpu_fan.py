"""The exact Siddon pair on fan planes at the sizes where its tiles, tables and
dealing can go wrong: volumes below, at and one past the 16-column blocks and
the 52-cell block height, detectors with fewer and more rows than a wavefront,
coarse to fine rows (the adjoint's row spacing), views along the grid axes
(paths that cross a face slowly), near 45 degrees, flat and cylindrical,
helical.  Tolerances are the pair's own: 1e-5 against the FP64 oracle, 1e-6
for the transpose."""
import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"


def _geometry(name):
    import nefct_hip as nh
    V, F = nh.VolumeGeometry, nh.ConeGeometry.flat
    return {
        "one-block": (V.cube((16, 16, 52), 1.0), F(200.0, 320.0, 40, 0.9, 64, 1.6), 9),
        "one-past": (V.cube((17, 33, 53), 1.0), F(200.0, 320.0, 61, 1.1, 65, 1.7), 9),
        "thin": (V((31, 15, 1), (1.0, -2.0, 0.3), (31.0, 15.0, 1.0)), F(150.0, 200.0, 37, 1.3, 3, 0.9), 7),
        "column": (V((1, 1, 110), (0.4, 0.2, 0.0), (1.0, 1.0, 110.0)), F(400.0, 600.0, 5, 1.0, 130, 1.4), 5),
        "fine-rows": (V.cube((20, 18, 12), 2.0), F(150.0, 260.0, 33, 2.1, 150, 0.4), 6),
        "coarse-rows": (V.cube((48, 40, 60), 0.5), F(150.0, 260.0, 50, 0.9, 9, 6.0), 8),
        "axis-views": (V.cube((40, 40, 24), 1.0), F(500.0, 800.0, 90, 0.8, 30, 1.3, ai=0.3), 4),
        "diagonal-views": (V.cube((40, 40, 24), 1.0), F(500.0, 800.0, 90, 0.8, 30, 1.3, ai=0.3), -4),
        "cyli": (V.cube((35, 37, 30), 1.2), nh.ConeGeometry("cyli", 120.0, 210.0, 67, 0.009, 0.4, 41, 1.7, 0.6), 8),
    }[name]


@pytest.mark.parametrize("name", ["one-block", "one-past", "thin", "column", "fine-rows", "coarse-rows", "axis-views",
                                  "diagonal-views", "cyli"])
def test_pair_against_oracle(oracle, name):
    import nefct_hip as nh
    vol, det, nv = _geometry(name)
    if abs(nv) == 4:    # within 1/50 rad of the grid axes / of the diagonals
        ang = (np.arange(16) % 4 * (math.pi / 2) + (math.pi / 4 if nv < 0 else 0.0)
               + np.linspace(-0.02, 0.02, 16)).astype(np.float32)
    else:
        ang = (2 * math.pi * np.arange(nv) / nv + 0.11).astype(np.float32)
    rng = np.random.default_rng(5)
    x = rng.uniform(0, 1, vol.shape_zyx).astype(np.float32)
    y = rng.uniform(0, 1, (ang.size, det.nb, det.na)).astype(np.float32)
    ov = oracle.vol_struct(vol.grid, vol.center, vol.size)
    od = oracle.det_struct(det.cyl, det.SID, det.SAD, det.na, det.da, det.ai, det.nb, det.db, det.bi)
    a = torch.tensor(ang)
    p = nh.project(torch.tensor(x, device=DEV), vol, det, a).double().cpu().numpy()
    b = nh.backproject(torch.tensor(y, device=DEV), vol, det, a).double().cpu().numpy()
    rp = oracle.exact_fwd(ov, od, ang.astype(np.float64), x.astype(np.float64))
    rb = oracle.exact_bp(ov, od, ang.astype(np.float64), y.astype(np.float64))
    assert np.linalg.norm(p - rp) <= 1e-5 * np.linalg.norm(rp)
    assert np.linalg.norm(b - rb) <= 1e-5 * np.linalg.norm(rb)
    lhs, rhs = float((p * y).sum()), float((b * x).sum())
    assert abs(lhs - rhs) <= 1e-6 * abs(lhs)


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_non_finite_voxel_reaches_only_its_rays(value):
    """A ray's sum is non-finite exactly where its length in the voxel is
    positive (the kernel reads two cells per piece, one of them perhaps
    without any length)."""
    import nefct_hip as nh
    vol, det, _ = _geometry("one-past")
    ang = torch.linspace(0.1, 6.0, 7)
    x = torch.rand(vol.shape_zyx, generator=torch.Generator().manual_seed(1)).to(DEV)
    one = torch.zeros_like(x)
    clean = nh.project(x, vol, det, ang)
    x[20, 11, 9] = value
    one[20, 11, 9] = 1.0
    hit = nh.project(one, vol, det, ang) > 0
    got = nh.project(x, vol, det, ang)
    assert hit.any() and torch.equal(torch.isfinite(got), ~hit)
    assert torch.equal(got[~hit], clean[~hit])


@pytest.mark.parametrize("signed", [False, True])
def test_split_views_add_the_same_bits(signed):
    """A volume of few blocks has its views split over workgroups (integer sums
    in the workspace); without a workspace they are not: the same bits."""
    import ctypes
    import nefct_hip as nh
    from nefct_hip import _lib
    from nefct_hip.ops import _ptr, _stream_ptr
    vol, det = nh.VolumeGeometry.cube((30, 20, 70), 1.0), nh.ConeGeometry.flat(150.0, 230.0, 50, 1.0, 81, 1.5)
    ang = torch.linspace(0, 6.2, 133, device=DEV)
    y = torch.rand((133, det.nb, det.na), generator=torch.Generator().manual_seed(2)).to(DEV) - (0.5 if signed else 0.0)
    want = torch.full(vol.shape_zyx, float("nan"), device=DEV)
    st = _lib.load().nefct_backproject_flat_noalloc(
        _ptr(y), _lib.int3(vol.grid), _lib.float3(vol.center), _lib.float3(vol.size), _ptr(ang), 133, det.SID, det.SAD,
        det.na, det.da, det.ai, det.nb, det.db, det.bi, _ptr(want), 0, ctypes.c_void_p(_stream_ptr(y.device)))
    _lib.check(st, "noalloc")
    assert torch.equal(nh.backproject(y, vol, det, ang), want)


def test_batch_of_both_walks_and_other_rule():
    """A batch of one fan-plane problem and one too steep for it equals the
    plain calls, also when called with the reference's rule after a plan for
    the exact one."""
    import nefct_hip as nh
    from nefct_hip import _lib
    from nefct_hip.batch import SiddonBatch
    steep = (nh.VolumeGeometry.cube((24, 24, 24), 1.0), nh.ConeGeometry.flat(30.0, 45.0, 12, 4.0, 40, 6.0),
             np.linspace(0, 5, 6).astype(np.float32))
    flat = (nh.VolumeGeometry.cube((20, 25, 30), 1.0), nh.ConeGeometry.flat(200.0, 320.0, 45, 1.1, 40, 1.7),
            np.linspace(0, 5, 9).astype(np.float32))
    b = SiddonBatch([flat, steep, flat])
    assert [p.pad_ for p in b.host] == [1, 0, 1]
    g = torch.Generator().manual_seed(3)
    xs = [torch.rand(v.shape, generator=g).to(DEV) for v in b.volumes]
    ys = [torch.rand(s.shape, generator=g).to(DEV) for s in b.sinograms]
    for fwd, adj in ((0, 0), (_lib.REF_FORWARD, _lib.REF_ADJOINT)):
        for v, x in zip(b.volumes, xs):
            v.copy_(x)
        b.flags = fwd
        b.project()
        for s, x, (vol, det, a) in zip(b.sinograms, xs, (flat, steep, flat)):
            ref = nh.project(x, vol, det, torch.tensor(a), flags=fwd)
            assert torch.allclose(s, ref, rtol=1e-6, atol=1e-6 * ref.abs().max().item())
        for s, y in zip(b.sinograms, ys):
            s.copy_(y)
        b.flags = adj
        b.backproject()
        for v, y, (vol, det, a) in zip(b.volumes, ys, (flat, steep, flat)):
            ref = nh.backproject(y, vol, det, torch.tensor(a), flags=adj)
            assert torch.allclose(v, ref, rtol=1e-6, atol=1e-6 * ref.abs().max().item())


@pytest.mark.parametrize("tilt", [0.0, 1e-7, 1e-5, 1e-3, 6e-3])
def test_slow_paths_along_faces(tilt):
    """Columns whose path runs along a cell face (every slab then has both of
    its parts, the fullest tables) or crosses one slowly, with rays that leave
    the volume in z: forward and adjoint see the same crossings."""
    import nefct_hip as nh
    vol = nh.VolumeGeometry.cube((48, 48, 40), 1.0)
    det = nh.ConeGeometry.flat(300.0, 450.0, 65, 1.5, 70, 1.5)       # column 32 looks along x = 0
    ang = torch.tensor([k * math.pi / 2 + s * tilt for k in range(4) for s in (1, -1)], dtype=torch.float32)
    g = torch.Generator().manual_seed(4)
    x = torch.rand(vol.shape_zyx, generator=g).to(DEV)
    y = torch.rand((8, det.nb, det.na), generator=g).to(DEV)
    p = nh.project(x, vol, det, ang)
    b = nh.backproject(y, vol, det, ang)
    lhs, rhs = (p.double() * y.double()).sum().item(), (x.double() * b.double()).sum().item()
    assert abs(lhs - rhs) <= 1e-6 * abs(lhs)
    # a constant volume gives the chords, which no choice of crossing changes
    ones = nh.project(torch.ones_like(x), vol, det, ang).double()
    lo, hi = ones[:, 35, 32].min().item(), ones[:, 35, 32].max().item()
    assert 48.0 * (1 - 1e-5) <= lo and hi <= 48.0 * (1 + 1e-3)
