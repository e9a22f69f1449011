"""Chained steps through the tiled x-forward (N1 past the short lines of the side-by-side one): forced against the oracle,
and after every other use of the state's buffers.

Tolerance: 1e-12 (FP64) and 1e-5 (FP32) of the largest value, as in the other step tests; the forced FP32 inputs are
checked to be ones whose result is determined that far (the oracle's step from inputs that differ by one part in 1e7
moves by less than a tenth of it)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pyoracle import Oracle  # noqa: E402


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available(), "GPU test run without a GPU"
    from tarang_amd import Context
    return Context(0)


def far(got, ref):
    m = max(np.abs(r).max() for r in ref)
    return max(np.abs(g - r).max() for g, r in zip(got, ref)) / m


def host(fields):
    return [f.cpu().numpy().astype(np.complex128) for f in fields]


@pytest.mark.parametrize("N", [(192, 64, 128), (256, 128, 64)])
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-5)])
def test_forced_step_and_last_stage(ctx, N, prec, tol):
    from tarang_amd import Plan, State
    print(N, prec, flush=True)
    nu, dt, force = 0.01, 1e-3, (1, 1.5, 3.5, 0.5, 0.3)
    o, p = Oracle(N), Plan(ctx, N, precision=prec)
    d = [p.to_dev(v) for v in o.ic_random(8, E0=0.5, kp=3.0)]
    V = host(d)
    if prec == "fp32":
        W = [v * (1 + 1e-7) for v in V]
        U = [v.copy() for v in V]
        o.step_ns_forced(W, nu, dt, *force, steps=2)
        o.step_ns_forced(U, nu, dt, *force, steps=2)
        assert far(W, U) < 0.1 * tol
    s = State(p)
    s.upload(d)
    s.set_force(*force)
    last = o.zeros(3)
    o.step_ns_forced(V, nu, dt, *force, steps=2, last_stage=last)
    s.step(dt, nu=nu, steps=2)
    assert far(host(s.download()), V) <= tol
    assert far(host(s.download_buffer(1)), last) <= tol


@pytest.mark.parametrize("forced", (False, True))
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-5)])
def test_ns_step_after_other_uses_of_the_state(ctx, prec, tol, forced):
    from tarang_amd import Plan, State
    N, nu, dt, force = (192, 24, 32), 0.01, 2e-3, (1, 1.5, 3.5, 0.2, 0.1)
    print(N, prec, forced, flush=True)
    o, p = Oracle(N), Plan(ctx, N, precision=prec)
    s = State(p)
    if forced:
        s.set_force(*force)
    V = []

    def upload(seed):
        d = [p.to_dev(v) for v in o.ic_random(seed)]
        V[:] = host(d)
        s.upload(d)

    def step_and_check(what):
        if prec == "fp32":
            V[:] = host(s.download())          # each step from what the state holds: no error carried over
        s.step(dt, nu=nu, steps=1)
        if forced:
            o.step_ns_forced(V, nu, dt, *force, steps=1)
        else:
            o.rk4_ns(V, nu, dt, steps=1)
        assert far(host(s.download()), V) <= tol, what

    upload(13)
    step_and_check("first")
    step_and_check("second")
    upload(14)
    step_and_check("upload")
    s.flux_shell_tr(np.concatenate([np.arange(6, dtype=float), [10000.0]]))
    step_and_check("flux")
    for stage in (1, 2, 3, 4):
        s.profile_passes(dt, nu=nu, stage=stage, nrep=1)
    step_and_check("profile")
    s.tune(dt, nu=nu, nrep=1)
    step_and_check("tune")
    s.set_force(*(force if not forced else (0, 0, 0, 0, 0)))
    forced = not forced
    step_and_check("forcing switched")


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-5)])
def test_mhd_step_after_other_uses_of_the_state(ctx, prec, tol):
    from tarang_amd import Plan, State, abi
    N, nu, eta, dt = (192, 16, 24), 0.01, 0.02, 2e-3
    print(N, prec, flush=True)
    o, p = Oracle(N), Plan(ctx, N, precision=prec)
    s = State(p, abi.TH_MHD)
    F = []

    def upload(seed):
        d = [p.to_dev(v) for v in o.ic_random(seed) + o.ic_random(seed + 1)]
        F[:] = host(d)
        s.upload(d)

    def step_and_check(what):
        if prec == "fp32":
            F[:] = host(s.download())
        s.step(dt, nu=nu, eta=eta, steps=1)
        o.rk4_mhd(F[:3], F[3:], nu, eta, dt, steps=1)
        assert far(host(s.download()), F) <= tol, what

    upload(21)
    step_and_check("first")
    step_and_check("second")
    upload(23)
    step_and_check("upload")
    s.flux_mhd(np.concatenate([np.arange(5, dtype=float), [10000.0]]))
    step_and_check("flux")
    for stage in (1, 2, 3, 4):
        s.profile_passes(dt, nu=nu, eta=eta, stage=stage, nrep=1)
    step_and_check("profile")
    s.tune(dt, nu=nu, eta=eta, nrep=1)
    step_and_check("tune")
