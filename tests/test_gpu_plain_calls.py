"""Calls of the plain steppers whose arguments or results the fused passes must treat as the separate operations do."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available(), "GPU test run without a GPU"
    from tarang_amd import Context
    return Context(0)


def _random(p, n, seed):
    import torch
    g = torch.Generator().manual_seed(seed)
    return [p.dealias(torch.view_as_complex(torch.randn(*p.shape, 2, generator=g, dtype=torch.float64)).mul_(0.05)
                      .to(p.dtype).cuda()) for _ in range(n)]


@pytest.mark.parametrize("physics", ("ns", "mhd"))
@pytest.mark.parametrize("scheme", (0, 1, 2))
def test_last_stage_may_be_the_fields_themselves(ctx, physics, scheme):
    """A program that does not need the last stage's input may give the fields' own arrays for it: they end as the step's
    result, the same bits as without it."""
    from tarang_amd import Plan
    print(physics, scheme, flush=True)
    p = Plan(ctx, (16, 24, 32))
    F = _random(p, 3 if physics == "ns" else 6, 3)
    a, b = [f.clone() for f in F], [f.clone() for f in F]
    for f, last in ((a, None), (b, b)):
        if physics == "ns":
            p.step_plain_forced(f, 2e-3, 3e-3, 1, 1.0, 3.0, 0.4, 0.1, scheme=scheme, last_stage=last)
        else:
            p.step_plain_forced_mhd(f[:3], f[3:], 2e-3, 3e-3, 5e-3, 1.0, 3.0, 0.4, 0.1, 0.1, 0.2, scheme=scheme,
                                    last_stage=last)
    for x, y in zip(a, b):
        assert np.array_equal(x.cpu().numpy(), y.cpu().numpy())


@pytest.mark.parametrize("scheme", (0, 1, 2))
def test_pure_decay_has_the_factor_of_exp_ksqr(ctx, scheme):
    """A shear flow (0, f(x), 0) has no nonlinear term, exactly (V_x = 0 and Ky = Kz = 0 on its modes): an EULER or RK4
    step multiplies each mode by exp(-nu K^2 dt), evaluated and rounded once, as exp_ksqr does; RK2 by the half step's
    factor twice."""
    import torch
    from tarang_amd import Plan, abi
    print(scheme, flush=True)
    nu, dt = 3e-3, 0.37
    p = Plan(ctx, (96, 16, 16), kfactor=(0.7, 1.0, 1.0))
    V = [torch.zeros(p.shape, dtype=p.dtype, device="cuda") for _ in range(3)]
    for k in range(1, 32):
        V[1][k, 0, 0] = complex(0.3 / k, 0.1)
        V[1][-k, 0, 0] = complex(0.3 / k, -0.1)
    ref = p.exp_ksqr(V[1].clone(), -nu * dt * (0.5 if scheme == 1 else 1.0))
    if scheme == 1:
        ref = p.exp_ksqr(ref, -nu * dt * 0.5)
    got = p.step_plain(abi.TH_NS, V, dt, nu=nu, scheme=scheme)[1]
    assert np.array_equal(got[:, 0, 0].cpu().numpy(), ref[:, 0, 0].cpu().numpy())
