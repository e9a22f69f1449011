"""Every line length on every axis: the array transforms against numpy's FFT, and one fused RK4 step against the
FP64 oracle, so that each radix schedule of each pass is run.

Tolerances: a transform of a line of L points has an error of about eps log2 L per stage on each of three axes, below
30 eps of the largest value for L <= 512: 1e-14 in FP64, 5e-6 in FP32; a step adds products and three more
transforms, 1e-12 and 1e-5 of the largest value as in the other step tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pyoracle import Oracle  # noqa: E402

LENGTHS = (24, 32, 48, 64, 96, 128, 192, 256, 384, 512)


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available(), "GPU test run without a GPU"
    from tarang_amd import Context
    return Context(0)


@pytest.mark.parametrize("L", LENGTHS)
@pytest.mark.parametrize("axis", (0, 1, 2))
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-14), ("fp32", 5e-6)])
def test_transforms_of_every_length(ctx, L, axis, prec, tol):
    from tarang_amd import Plan
    N = [8, 8, 8]
    N[axis] = L
    print(N, prec, flush=True)
    p = Plan(ctx, N, precision=prec)
    u = np.random.default_rng(L + axis).standard_normal(N)
    packed = np.zeros(p.shape, np.complex128)
    packed[:, :, :-1] = u[:, :, 0::2] + 1j * u[:, :, 1::2]
    ref = np.fft.rfftn(u, norm="forward")
    d = p.to_dev(packed)
    p.forward(d)
    assert np.abs(d.cpu().numpy() - ref).max() <= tol * np.abs(ref).max()
    d = p.to_dev(np.ascontiguousarray(ref))
    p.inverse(d)
    assert np.abs(d.cpu().numpy() - packed).max() <= tol * np.abs(packed).max()


@pytest.mark.parametrize("L", LENGTHS)
@pytest.mark.parametrize("axis", (0, 1, 2))
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-5)])
def test_fused_step_of_every_length(ctx, L, axis, prec, tol):
    from tarang_amd import Plan, State
    N = [16, 16, 16]
    N[axis] = L
    print(N, prec, flush=True)
    o = Oracle(N)
    V = o.ic_random(7, E0=0.5, kp=3.0)
    p = Plan(ctx, N, precision=prec)
    s = State(p)
    s.upload([p.to_dev(v) for v in V])
    s.step(2e-3, nu=5e-3, steps=2)
    o.rk4_ns(V, 5e-3, 2e-3, steps=2)
    m = max(np.abs(v).max() for v in V)
    for got, ref in zip(s.download(), V):
        assert np.abs(got.cpu().numpy() - ref).max() <= tol * m
