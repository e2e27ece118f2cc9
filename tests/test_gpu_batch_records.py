"""A batch whose column records take several turns of their grid: many small
problems and one with more views and columns than the grid has blocks for."""
import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"


def test_one_long_wide_problem_among_many():
    import nefct_hip as nh
    from nefct_hip.batch import SiddonBatch
    small = (nh.VolumeGeometry.cube((8, 8, 8), 1.0), nh.ConeGeometry.flat(200.0, 300.0, 16, 0.8, 16, 0.8),
             np.linspace(0.1, 3.0, 4).astype(np.float32))
    big = (nh.VolumeGeometry.cube((16, 16, 16), 1.0), nh.ConeGeometry.flat(200.0, 300.0, 1300, 0.02, 32, 0.8),
           (0.1 + 2 * math.pi * np.arange(90) / 90).astype(np.float32))
    probs = [small] * 150 + [big] + [small] * 50
    b = SiddonBatch(probs, device=DEV)
    assert {p.pad_ for p in b.host} <= {1, 3}       # adjoints on fan planes
    g = torch.Generator().manual_seed(9)
    at = (0, 149, 150, 151, 200)
    for v in b.volumes:
        v.copy_(torch.rand(v.shape, generator=g))
    xs = {i: b.volumes[i].clone() for i in at}
    b.project()
    for i in at:
        vol, det, ang = probs[i]
        ref = nh.project(xs[i], vol, det, torch.tensor(ang))
        assert torch.allclose(b.sinograms[i], ref, rtol=1e-6, atol=1e-6 * ref.abs().max().item()), i
    for s in b.sinograms:
        s.copy_(torch.rand(s.shape, generator=g))
    ys = {i: b.sinograms[i].clone() for i in at}
    b.backproject()
    for i in at:
        vol, det, ang = probs[i]
        assert torch.equal(b.volumes[i], nh.backproject(ys[i], vol, det, torch.tensor(ang))), i


def test_batch_of_all_four_walks():
    """Problems walked per ray, on fan planes, and so in one direction only, in
    one batch; also called with the reference's rule after a plan for the exact
    one."""
    import nefct_hip as nh
    from nefct_hip import _lib
    from nefct_hip.batch import SiddonBatch
    F = nh.ConeGeometry.flat
    ang = {n: (0.2 + 2 * math.pi * np.arange(n) / n).astype(np.float32) for n in (6, 9, 12, 60)}
    probs = [
        (nh.VolumeGeometry.cube((24, 24, 24), 1.0), F(30.0, 45.0, 12, 4.0, 40, 6.0), ang[6]),           # steep
        (nh.VolumeGeometry.cube((20, 25, 30), 1.0), F(200.0, 320.0, 45, 1.1, 40, 1.7), ang[9]),
        (nh.VolumeGeometry.cube((64, 64, 1), 1.0), F(1000.0, 1500.0, 128, 0.75, 1, 1.5, bi=0.55), ang[12]),
        (nh.VolumeGeometry.cube((120, 130, 90), 1.0), F(1000.0, 1500.0, 240, 0.81, 45, 3.1, bi=0.55), ang[60]),
    ]
    b = SiddonBatch(probs, device=DEV)
    assert [p.pad_ for p in b.host] == [0, 1, 2, 3]
    g = torch.Generator().manual_seed(11)
    xs = [torch.rand(v.shape, generator=g).to(DEV) for v in b.volumes]
    ys = [torch.rand(s.shape, generator=g).to(DEV) for s in b.sinograms]
    for fwd, adj in ((0, 0), (_lib.REF_FORWARD, _lib.REF_ADJOINT)):
        for v, x in zip(b.volumes, xs):
            v.copy_(x)
        b.flags = fwd
        b.project()
        for s, x, (vol, det, a) in zip(b.sinograms, xs, probs):
            ref = nh.project(x, vol, det, torch.tensor(a), flags=fwd)
            assert torch.allclose(s, ref, rtol=1e-6, atol=1e-6 * ref.abs().max().item())
        for s, y in zip(b.sinograms, ys):
            s.copy_(y)
        b.flags = adj
        b.backproject()
        for v, y, (vol, det, a) in zip(b.volumes, ys, probs):
            assert torch.equal(v, nh.backproject(y, vol, det, torch.tensor(a), flags=adj))
