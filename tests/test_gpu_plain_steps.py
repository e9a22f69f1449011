"""The plain steppers through the fused passes against the same step put together from the array operations
(nlin, pressure, rhs, compute_force) on fields of every mode, dealiased or not: all schemes, physics, forces, both
precisions, anisotropic factors, lengths of both kinds; and the calls that stay on the operation sequence.

Tolerance: a step is three to five transforms and a few sums per mode; 1e-12 (FP64) and 1e-5 (FP32) of the largest
value, as in the other step tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DT, D0, D1 = 2e-3, 3e-3, 5e-3


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available(), "GPU test run without a GPU"
    from tarang_amd import Context
    return Context(0)


def _rhs(p, physics, F, force):
    G = [f.clone() for f in F]
    if physics == "ns":
        n = p.nlin_ns(G)
        if force is not None:
            n = [a - b for a, b in zip(n, force(F))]
        return p.rhs(n, p.pressure(n))
    if physics == "mhd":
        FF = force(F) if force is not None else None
        n, nb = p.nlin_mhd(G[:3], G[3:])
        if FF is not None:
            n, nb = [a - b for a, b in zip(n, FF[:3])], [a - b for a, b in zip(nb, FF[3:])]
        return p.rhs(n, p.pressure(n)) + [-b for b in nb]
    n, nt = p.nlin_rb(G[:3], G[3])
    n[0] = n[0] - p.dealias(F[3].clone())
    nt = nt - p.dealias(F[0].clone())
    return p.rhs(n, p.pressure(n)) + [-nt]


def _step(p, physics, F, scheme, force):
    d = [D0] * 3 + [D1] * 3

    def E(x, c, a):                       # exp(-diss K^2 a dt) x
        return p.exp_ksqr(x.clone(), -d[c] * a * DT)
    if scheme == 0:
        r = _rhs(p, physics, F, force)
        out = [E(f + DT * a, c, 1) for c, (f, a) in enumerate(zip(F, r))]
    elif scheme == 1:
        r = _rhs(p, physics, F, force)
        v = [E(f + 0.5 * DT * a, c, 0.5) for c, (f, a) in enumerate(zip(F, r))]
        r = _rhs(p, physics, v, force)
        out = [E(E(f, c, 0.5) + DT * a, c, 0.5) for c, (f, a) in enumerate(zip(F, r))]
    else:
        r = _rhs(p, physics, F, force)
        acc = [DT / 6 * E(a, c, 1) for c, a in enumerate(r)]
        v = [E(f + 0.5 * DT * a, c, 0.5) for c, (f, a) in enumerate(zip(F, r))]
        r = _rhs(p, physics, v, force)
        acc = [t + DT / 3 * E(a, c, 0.5) for c, (t, a) in enumerate(zip(acc, r))]
        v = [E(f, c, 0.5) + 0.5 * DT * a for c, (f, a) in enumerate(zip(F, r))]
        r = _rhs(p, physics, v, force)
        acc = [t + DT / 3 * E(a, c, 0.5) for c, (t, a) in enumerate(zip(acc, r))]
        v = [E(E(f, c, 0.5) + DT * a, c, 0.5) for c, (f, a) in enumerate(zip(F, r))]
        r = _rhs(p, physics, v, force)
        out = [E(f, c, 1) + t + DT / 6 * a for c, (f, t, a) in enumerate(zip(F, acc, r))]
    return [p.dealias(f) for f in out]


def _fields(p, n, seed):
    import torch
    g = torch.Generator().manual_seed(seed)
    return [torch.view_as_complex(torch.randn(*p.shape, 2, generator=g, dtype=torch.float64)).mul_(0.05).to(p.dtype).cuda()
            for _ in range(n)]


# (grid, kfactor): smallest lengths, mixed ones, an x line of each schedule family
GRIDS = [((16, 16, 16), (1.0, 1.0, 1.0)), ((24, 32, 48), (1.0, 0.5, 2.0)), ((96, 16, 64), (1.0, 1.0, 1.0)),
         ((64, 192, 32), (2.0, 1.0, 0.5))]


@pytest.mark.parametrize("grid", GRIDS)
@pytest.mark.parametrize("physics", ("ns", "mhd", "rb"))
@pytest.mark.parametrize("scheme", (0, 1, 2))
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-5)])
def test_plain_step_equals_its_operations(ctx, grid, physics, scheme, prec, tol):
    from tarang_amd import Plan, abi
    N, kf = grid
    print(N, kf, physics, scheme, prec, flush=True)
    p = Plan(ctx, N, kfactor=kf, basis="SCFT" if physics == "rb" else "FOUR", precision=prec)
    F = _fields(p, {"ns": 3, "mhd": 6, "rb": 4}[physics], 11)
    ref = _step(p, physics, [f.clone() for f in F], scheme, None)
    got = p.step_plain({"ns": abi.TH_NS, "mhd": abi.TH_MHD, "rb": abi.TH_RB}[physics], F, DT, nu=D0, eta=D1, kappa=D1,
                       scheme=scheme)
    m = max(float(r.abs().max()) for r in ref)
    for a, b in zip(got, ref):
        assert float((a - b).abs().max()) <= tol * m


# bands inside the kept modes (fused passes) and reaching past them (operation sequence), fixed fields
@pytest.mark.parametrize("proc,inner,outer,p3", [(1, 1.0, 3.0, 0.4), (2, 1.0, 3.0, 0.02), (1, 2.0, 7.5, 0.4), (3, 2.0, 0.3, 0.2)])
@pytest.mark.parametrize("physics", ("ns", "mhd"))
@pytest.mark.parametrize("scheme", (0, 1, 2))
def test_forced_plain_step_equals_its_operations(ctx, proc, inner, outer, p3, physics, scheme):
    from tarang_amd import Plan
    N = (24, 16, 32)
    print(proc, inner, outer, physics, scheme, flush=True)
    p = Plan(ctx, N)
    F = _fields(p, 3 if physics == "ns" else 6, 5)
    p5, p6 = (0.1, 0.2) if proc != 3 else (0.0, 0.0)
    if physics == "ns":
        ref = _step(p, physics, [f.clone() for f in F], scheme, lambda V: p.compute_force(V, proc, inner, outer, p3, 0.1)[0])
        last = [f.clone() for f in F]
        got = p.step_plain_forced(F, DT, D0, proc, inner, outer, p3, 0.1, scheme=scheme, last_stage=last)
    else:
        def force(V):
            fu, fw, _ = p.compute_force_mhd(V[:3], V[3:], proc, inner, outer, p3, 0.1, p5, p6)
            return fu + fw
        ref = _step(p, physics, [f.clone() for f in F], scheme, force)
        last = [f.clone() for f in F]
        u, b = p.step_plain_forced_mhd(F[:3], F[3:], DT, D0, D1, inner, outer, p3, 0.1, p5, p6, scheme=scheme, proc=proc,
                                       last_stage=last)
        got = list(u) + list(b)
    m = max(float(r.abs().max()) for r in ref)
    for a, b in zip(got, ref):
        assert float((a - b).abs().max()) <= 1e-12 * m
