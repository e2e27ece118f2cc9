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
