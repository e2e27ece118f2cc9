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
