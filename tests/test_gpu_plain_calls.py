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
