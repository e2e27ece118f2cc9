"""The warp's adjoint where neighbouring voxels hand corner sums to each other
(along x between lanes, along y from row to row) and where they must not:
smooth fields, jumps, random ones, samples without a value, rows and columns
at the edges of the lanes' share.  And the inverse of a displacement field
that comes to rest, and of one that alternates between two states."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"


def _field(kind, shape, rng):
    nz, ny, nx = shape
    z, y, x = np.meshgrid(*(np.arange(n, dtype=np.float32) for n in shape), indexing="ij")
    if kind == "smooth":
        m = [1.3 * np.sin(0.11 * x + 0.07 * y + k) + 0.4 * np.cos(0.2 * z + k) for k in range(3)]
    elif kind == "jump":
        m = [np.where((x > nx // 2) ^ (y > 2), 2.25, -1.5) + 0.0 * z for _ in range(3)]
    else:
        m = [rng.uniform(-3, 3, shape) for _ in range(3)]
    return np.stack(m).astype(np.float32)


def _scatter(g, m, boundary):
    """Transpose of the trilinear warp and the same of |g|, in FP64."""
    nz, ny, nx = g.shape
    z, y, x = np.meshgrid(*(np.arange(n, dtype=np.float32) for n in g.shape), indexing="ij")
    p = [x + m[0], y + m[1], z + m[2]]
    fin = np.isfinite(m).all(0)
    lo = [np.where(fin, np.floor(q), -9).astype(np.int64) for q in p]
    f = [np.where(fin, q - np.floor(q), 0).astype(np.float64) for q in p]
    n = (nx, ny, nz)
    ok = fin.copy()
    if boundary == 0:
        for a in range(3):
            ok &= (lo[a] > 0) & (lo[a] + 1 < n[a])
    out, mag = np.zeros(g.size), np.zeros(g.size)
    for q in range(8):
        c = [lo[a] + ((q >> a) & 1) for a in range(3)]
        w = np.prod([f[a] if (q >> a) & 1 else 1.0 - f[a] for a in range(3)], axis=0)
        s = ok & np.all([(c[a] >= 0) & (c[a] < n[a]) for a in range(3)], axis=0)
        i = (c[0] + nx * (c[1] + ny * c[2]))[s]
        np.add.at(out, i, (g.astype(np.float64) * w)[s])
        np.add.at(mag, i, np.abs(g.astype(np.float64) * w)[s])
    return out.reshape(g.shape), mag.reshape(g.shape)


@pytest.mark.parametrize("boundary", [0, 1])
@pytest.mark.parametrize("kind", ["smooth", "jump", "random"])
@pytest.mark.parametrize("shape", [(3, 1, 1), (4, 4, 63), (5, 5, 64), (4, 7, 65), (3, 9, 257)])
def test_adjoint_exchange(shape, kind, boundary):
    from nefct_hip.deform import deform_adjoint_op
    rng = np.random.default_rng(17)
    m = _field(kind, shape, rng)
    g = rng.standard_normal(shape).astype(np.float32)
    g[rng.random(shape) < 0.1] = 0.0
    m[0][rng.random(shape) < 0.03] = np.nan
    t = [torch.tensor(a, device=DEV) for a in (g, *m)]
    got = deform_adjoint_op(*t, boundary).double().cpu().numpy()
    want, mag = _scatter(g, m, boundary)
    # FP32 sums of some tens of products: 4e-6 of the summed magnitudes
    assert np.all(np.abs(got - want) <= 4e-6 * mag + 1e-30)


@pytest.mark.parametrize("iters", [0, 1, 2, 3, 6, 7, 30])
def test_invert_stops_on_the_right_state(oracle, iters):
    """x -> -(i + x - c) alternates between 0 and c - i wherever the sample
    stays in the volume; the other half of the volume comes to rest."""
    from nefct_hip.deform import invert_dvf
    nz, ny, nx = 4, 6, 16
    m = np.zeros((3, nz, ny, nx), np.float32)
    m[0, :2] = np.arange(nx, dtype=np.float32) - 8.0
    m[1, 2:] = 0.25 * np.sin(np.arange(ny, dtype=np.float32))[None, :, None]
    inv = invert_dvf(*(torch.tensor(a, device=DEV) for a in m), iters).cpu().numpy()
    want = oracle.invert_dvf(*m, iters=iters)
    for k in range(3):
        assert np.max(np.abs(inv[k] - want[k])) < 1e-5


@pytest.mark.parametrize("boundary", [0, 1])
@pytest.mark.parametrize("shape", [(4, 11, 17), (3, 9, 64), (3, 10, 130)])
def test_adjoint_of_rows_on_voxels_between_others(shape, boundary):
    """Rows whose samples all lie on voxels (displacements of 0, 1 and -2) or
    have no gradient hand nothing on; the rows around them do."""
    from nefct_hip.deform import deform_adjoint_op
    rng = np.random.default_rng(5)
    m = _field("smooth", shape, rng)
    g = rng.standard_normal(shape).astype(np.float32)
    for y, d in ((1, 0.0), (2, 1.0), (5, -2.0), (8, 0.0)):
        m[:, :, y] = d
    g[:, 6] = 0.0
    t = [torch.tensor(a, device=DEV) for a in (g, *m)]
    got = deform_adjoint_op(*t, boundary).double().cpu().numpy()
    want, mag = _scatter(g, m, boundary)
    # FP32 sums of some tens of products: 4e-6 of the summed magnitudes
    assert np.all(np.abs(got - want) <= 4e-6 * mag + 1e-30)
