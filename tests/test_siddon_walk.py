"""Which kernels a Siddon call takes (host code, no GPU): the fan-plane ones only
where they apply and pay."""
import os

import pytest


def walk(grid, na, nb, nv, da, db, voxel=1.0, SID=1000.0, SAD=1500.0, cyl=0, flags=0, adjoint=0, center=(0, 0, 0)):
    from nefct_hip import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    size = [n * voxel for n in grid]
    return _lib.load().nefct_siddon_walk(_lib.int3(grid), _lib.float3(center), _lib.float3(size), nv, SID, SAD, na,
                                         da, 0.5, nb, db, 0.5, cyl, flags, adjoint)


C1 = dict(grid=(128, 128, 128), na=256, nb=256, nv=180, da=1.5, db=1.5)


def test_variants_of_the_adjoint_that_keep_their_own_kernels():
    from nefct_hip import _lib as L
    for flags, fan in ((0, 1), (L.F_DETERMINISTIC, 1), (L.F_ADJ_FLOAT_ATOMIC, 1), (L.F_TILE_64x32x8, 1),
                       (L.F_ADJ_WINDOW, 0), (L.F_ADJ_FLOAT_ATOMIC | L.F_DETERMINISTIC, 0), (L.REF_ADJOINT, 0)):
        assert walk(**C1, flags=flags, adjoint=1) == fan, hex(flags)
        # the forward knows none of the adjoint's variants
        assert walk(**C1, flags=flags, adjoint=0) == (0 if flags & L.F_REF_SLAB else 1), hex(flags)


def test_steep_cones_and_bad_geometry():
    assert walk((64, 64, 64), 128, 128, 30, 1.0, 2.0, SID=77.0, SAD=115.0) == 0
    assert walk((64, 64, 64), 128, 128, 30, 1.0, 2.0, SID=77.0, SAD=115.0, adjoint=1) == 0
    assert walk((64, 64, 0), 128, 128, 30, 1.0, 1.0) == -2
    assert walk((64, 64, 64), 128, 128, 30, 1.0, 1.0, SID=-5.0) == -3


# scans timed with both walks, us of the forward / the adjoint on fan planes and
# per ray (the adjoint unsplit where the volume has few blocks)
@pytest.mark.parametrize("grid, na, nb, nv, db, forward, adjoint", [
    ((128, 128, 128), 256, 256, 180, 1.5, 1, 1),        # 330 / 410, 545 / 1313
    ((512, 512, 256), 1024, 768, 720, 0.6, 1, 1),       # 76 / 97, 181 / 263 ms
    ((32, 32, 32), 64, 48, 12, 6.0, 1, 1),              # 29 / 33
    ((512, 512, 8), 1024, 8, 150, 1.5, 0, 0),           # 1768 / 588, 1900 / 886
    ((512, 512, 1), 1024, 1, 150, 1.5, 0, 0),           # 1513 / 399, 2493 / 801
    ((512, 512, 48), 1024, 48, 150, 1.5, 0, 1),         # 2560 / 1991, 3729 / 4126
    ((512, 512, 65), 1024, 65, 150, 1.5, 0, 1),         # 4379 / 2732, 5628 / 6020
    ((256, 256, 16), 512, 64, 60, 0.375, 1, 1),         # 209 / 334, 477 / 1090 (rows a quarter of a voxel apart)
    ((256, 256, 256), 512, 16, 60, 24.0, 0, 1),         # 613 / 271, 925 / 1259 (sixteen voxels apart)
    ((318, 318, 202), 795, 146, 360, 2.08, 0, 1),       # 16991 / 6967, 16547 / 16027
    ((128, 128, 4), 256, 4, 180, 1.5, 0, 1),            # 162 / 88, 174 / 904: 16 blocks would leave the chip idle
    ((96, 96, 16), 192, 64, 60, 0.375, 1, 1),           # 45 / 69
])
def test_the_faster_walk(grid, na, nb, nv, db, forward, adjoint):
    voxel = 0.8 if grid == (512, 512, 256) else 4.0 if grid[0] == 32 else 1.0
    da = 0.6 if grid == (512, 512, 256) else 6.0 if grid[0] == 32 else max(grid[0] * 1.5 / na, 1.5 * (na == 256))
    assert walk(grid, na, nb, nv, da, db, voxel) == forward
    assert walk(grid, na, nb, nv, da, db, voxel, adjoint=1) == adjoint


def test_a_volume_beside_the_detector_and_a_cylinder():
    assert walk((64, 64, 8), 128, 8, 90, 0.75, 1.5, center=(0, 0, 500.0)) in (0, 1)
    flat = walk((512, 512, 64), 1024, 64, 150, 0.75, 3.0)
    assert flat == walk((512, 512, 64), 1024, 64, 150, 0.75 / 1500.0, 3.0, cyl=1) == 0


def test_batch_plans_count_each_direction_by_its_walk():
    """(a table on the host alone: nothing is launched)"""
    import ctypes
    from nefct_hip import _lib
    from nefct_hip.batch import Problem
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    table = (Problem * 3)()
    shapes = [((512, 512, 8), 1024, 8, 0), ((512, 512, 48), 1024, 48, 3), ((128, 128, 128), 256, 256, 1)]
    for p, (grid, na, nb, _) in zip(table, shapes):
        p.volume = p.sinogram = p.angles = 4096      # never read
        p.grid = _lib.int3(grid)
        p.center, p.size = _lib.float3((0, 0, 0)), _lib.float3([float(n) for n in grid])
        p.nv, p.cyl, p.SID, p.SAD, p.na, p.nb = 150, 0, 1000.0, 1500.0, na, nb
        p.da, p.ai, p.db, p.bi = grid[0] * 1.5 / na, 0.5, 1.5, 0.5
    out = [ctypes.c_size_t(), ctypes.c_longlong(), ctypes.c_longlong()]
    assert _lib.load().nefct_batch_plan(ctypes.addressof(table), 3, 0, *[ctypes.addressof(o) for o in out]) == 0
    for p, (grid, na, nb, kind) in zip(table, shapes):
        assert p.pad_ == kind
        cols, rows = (4, 64) if kind == 1 else (16, 16)
        assert (p.tiles_a, p.tiles_b) == (-(-na // cols), -(-nb // rows))
        x, z = (16, 52) if kind else (32, 16)
        assert list(p.blocks) == [-(-grid[0] // x), -(-grid[1] // x), -(-grid[2] // z)]
    # the other rule's kernels for all of them
    assert _lib.load().nefct_batch_plan(ctypes.addressof(table), 3, _lib.REF_FORWARD,
                                        *[ctypes.addressof(o) for o in out]) == 0
    assert [p.pad_ for p in table] == [0, 0, 0]
