"""Total variation and squared norm where their workgroups sum several planes
and runs of four: plane counts that the workgroups' share does not divide, one
that holds the whole depth, the value with and without a gradient, lengths of
every remainder, and data that starts at any FP32 boundary."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu
DEV = "cuda"


# (33 x 2 workgroups of columns: 2 planes each, the last 1), (1025: all 3), (2: one each)
@pytest.mark.parametrize("shape", [(37, 130, 70), (3, 4100, 64), (5, 7, 3)])
def test_planes_per_workgroup(oracle, shape):
    from nefct_hip.recon import _tv_hip, tv_smooth
    eps = 0.05
    x = torch.rand(shape, generator=torch.Generator().manual_seed(2))
    xn = x.double().numpy()
    d = oracle.tv_forward(xn)
    r = np.sqrt(d * d + eps * eps)
    xa = x.to(DEV).requires_grad_(True)
    va = tv_smooth(xa, eps)
    va.backward()
    want = oracle.tv_adjoint(d / r)
    assert va.item() == pytest.approx(r.sum(), rel=1e-6)
    assert np.linalg.norm(xa.grad.double().cpu().numpy() - want) <= 1e-5 * np.linalg.norm(want)
    # both in one pass, scaled: the same terms
    v, g = _tv_hip(x.to(DEV), eps, 0.5, True, True)
    assert v.item() == pytest.approx(0.5 * r.sum(), rel=1e-6)
    assert np.linalg.norm(2.0 * g.double().cpu().numpy() - want) <= 1e-5 * np.linalg.norm(want)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 4095, 4097, 16386, 16387, 4 * 1024 * 512 + 1027])
@pytest.mark.parametrize("first", [0, 1, 2, 3])
def test_sq_norm_remainders(n, first):
    from nefct_hip.recon import _sq_norm_into
    x = torch.randn(n + first, generator=torch.Generator().manual_seed(n))
    want = 0.5 * float((x[first:].double() ** 2).sum())
    value = torch.zeros((), dtype=torch.float64, device=DEV)
    _sq_norm_into(x.to(DEV)[first:], value, 0.5)
    assert value.item() == pytest.approx(want, rel=1e-10)    # FP64 sums of exact squares


def test_gradient_alone_is_no_slower_than_the_step_that_contains_it():
    """The descent step reads one volume more than the gradient and computes the
    same; sharing planes between workgroups, which only the value's sum needs,
    made the gradient 1.5 times the step."""
    from nefct_hip.recon import _tv_hip, tv_descent_step
    x = torch.rand((192, 512, 512), generator=torch.Generator().manual_seed(3)).to(DEV)
    d = torch.zeros_like(x)

    def us(fn):
        fn()
        best = float("inf")
        for _ in range(5):
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record()
            for _ in range(5):
                fn()
            e[1].record()
            torch.cuda.synchronize()
            best = min(best, e[0].elapsed_time(e[1]) * 200.0)
        return best

    grad = us(lambda: _tv_hip(x, 1e-3, 1.0, False, True))
    step = us(lambda: tv_descent_step(x, d, 1e-3, 0.1, 0.1))
    assert grad <= 1.25 * step, (grad, step)
