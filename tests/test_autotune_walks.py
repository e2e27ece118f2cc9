"""The autotuner where candidates are names of one kernel: it is timed once, the
default's name is kept, and the record says which walk ran (CPU: the timing and
the projections are stood in for)."""
import os

import pytest


@pytest.fixture
def tuner(monkeypatch):
    from nefct_hip import _lib, autotune
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    ran = []

    def time_ms(fn, reps):
        ran.append(fn())
        return 5.0 + len(ran)
    monkeypatch.setattr(autotune, "_time_ms", time_ms)
    return autotune, ran


@pytest.mark.parametrize("adjoint", [True, False])
@pytest.mark.parametrize("steep", [False, True])
def test_alike_candidates_are_timed_once(tuner, adjoint, steep):
    import nefct_hip as nh
    at, ran = tuner
    vol = nh.VolumeGeometry.cube((64, 64, 64), 1.0)
    det = nh.ConeGeometry.flat(77.0, 115.0, 128, 1.0, 128, 2.0) if steep else \
        nh.ConeGeometry.flat(700.0, 1050.0, 128, 0.75, 128, 0.75)
    cands = at.ADJOINT_CANDIDATES if adjoint else at.FORWARD_CANDIDATES
    times = at._time_candidates(vol, det, 60, 0, cands, adjoint, lambda flags: flags, 1)
    assert list(times) == list(cands) and len(ran) == len(set(ran))
    if steep:
        assert len(ran) == len(cands)
    else:       # fixed sums, float sums and the windows; one per view group
        assert len(ran) == (3 if adjoint else len(at.FORWARD_VIEW_GROUPS))
    rec = at._record(vol, det, 60, 0, cands, times, adjoint, 60)
    assert rec["variant"] == list(cands)[0] and rec["walk"] == ("per ray" if steep else "fan planes")
    assert set(rec["ms_on_sample"]) == set(cands)


def test_walks_fan_planes_refuses_bad_geometry():
    import nefct_hip as nh
    from nefct_hip import autotune, _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    vol = nh.VolumeGeometry.cube((64, 64, 64), 1.0)
    with pytest.raises(nh.NefctError):
        autotune.walks_fan_planes(vol, nh.ConeGeometry.flat(-1.0, 115.0, 8, 1.0, 8, 1.0), 10, 0, False)
