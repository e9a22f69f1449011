"""The plain steppers through the fused passes at every line length on every axis, each against the same step put together
from the array operations (test_gpu_plain_steps), so that each length's x-inverse of reference-layout fields and each
full-width z pass is run in every physics; and the last stage's input that a forced step hands out.

Tolerance: as there, 1e-12 (FP64) and 1e-5 (FP32) of the largest value."""
import pytest

from test_gpu_plain_steps import D0, D1, DT, _fields, _rhs, _step

pytestmark = pytest.mark.gpu

LENGTHS = (24, 32, 48, 64, 96, 128, 192, 256, 384, 512)


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available(), "GPU test run without a GPU"
    from tarang_amd import Context
    return Context(0)


@pytest.mark.parametrize("L", LENGTHS)
@pytest.mark.parametrize("axis", (0, 1, 2))
@pytest.mark.parametrize("physics", ("ns", "mhd", "rb"))
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-5)])
def test_plain_step_of_every_length(ctx, L, axis, physics, prec, tol):
    from tarang_amd import Plan, abi
    if physics == "rb" and axis == 0 and L == 384:
        pytest.skip("the array transforms take no sine / cosine lines of 384 points")
    N = [16, 16, 16]
    N[axis] = L
    print(N, physics, prec, flush=True)
    p = Plan(ctx, N, basis="SCFT" if physics == "rb" else "FOUR", precision=prec)
    F = _fields(p, {"ns": 3, "mhd": 6, "rb": 4}[physics], 100 * axis + L)
    ref = _step(p, physics, [f.clone() for f in F], 2, None)
    got = p.step_plain({"ns": abi.TH_NS, "mhd": abi.TH_MHD, "rb": abi.TH_RB}[physics], F, DT, nu=D0, eta=D1, kappa=D1, scheme=2)
    m = max(float(r.abs().max()) for r in ref)
    for a, b in zip(got, ref):
        assert float((a - b).abs().max()) <= tol * m


@pytest.mark.parametrize("physics", ("ns", "mhd"))
@pytest.mark.parametrize("scheme", (0, 1, 2))
@pytest.mark.parametrize("outer", (3.0, 7.5))     # through the fused passes, and by the separate operations
def test_last_stage_is_the_input_of_the_last_stage(ctx, physics, scheme, outer):
    from tarang_amd import Plan
    print(physics, scheme, outer, flush=True)
    p = Plan(ctx, (24, 16, 32))
    F = _fields(p, 3 if physics == "ns" else 6, 5)

    def force(V):
        if physics == "ns":
            return p.compute_force(V, 1, 1.0, outer, 0.4, 0.1)[0]
        fu, fw, _ = p.compute_force_mhd(V[:3], V[3:], 1, 1.0, outer, 0.4, 0.1, 0.1, 0.2)
        return fu + fw

    def E(x, c, a):
        return p.exp_ksqr(x.clone(), -(D0 if c < 3 else D1) * a * DT)
    ref = [f.clone() for f in F]
    if scheme > 0:
        r = _rhs(p, physics, F, force)
        ref = [E(f + 0.5 * DT * a, c, 0.5) for c, (f, a) in enumerate(zip(F, r))]
    if scheme == 2:
        r = _rhs(p, physics, ref, force)
        ref = [E(f, c, 0.5) + 0.5 * DT * a for c, (f, a) in enumerate(zip(F, r))]
        r = _rhs(p, physics, ref, force)
        ref = [E(E(f, c, 0.5) + DT * a, c, 0.5) for c, (f, a) in enumerate(zip(F, r))]
    last = [f.clone() for f in F]
    if physics == "ns":
        p.step_plain_forced(F, DT, D0, 1, 1.0, outer, 0.4, 0.1, scheme=scheme, last_stage=last)
    else:
        p.step_plain_forced_mhd(F[:3], F[3:], DT, D0, D1, 1.0, outer, 0.4, 0.1, 0.1, 0.2, scheme=scheme, proc=1, last_stage=last)
    m = max(float(r.abs().max()) for r in ref)
    for a, b in zip(last, ref):
        assert float((a - b).abs().max()) <= 1e-12 * m
