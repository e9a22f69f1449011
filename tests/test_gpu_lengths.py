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


# the edges of the short-box rules: smallest planes, one row of every length of the plane pass, the largest planes of
# each precision, boxes on both sides of the split x-forward's line; boxes = 20 passes the group counts' limits
@pytest.mark.parametrize("N", [(16, 16, 16), (24, 24, 24), (32, 48, 32), (48, 96, 48), (256, 64, 128), (64, 128, 64),
                               (128, 16, 128), (96, 64, 64), (128, 96, 64), (256, 128, 64), (64, 128, 128)])
@pytest.mark.parametrize("physics", ("ns", "mhd", "rb"))
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-5)])
def test_short_boxes(ctx, N, physics, prec, tol):
    from tarang_amd import Plan, State, abi
    print(N, physics, prec, flush=True)
    basis = "SCFT" if physics == "rb" else "FOUR"
    o = Oracle(N, basis=basis)
    p = Plan(ctx, N, basis=basis, precision=prec)
    F = o.ic_random(7, E0=0.5, kp=3.0)
    F += o.ic_random(8, E0=0.3, kp=3.0) if physics == "mhd" else [o.ic_random_scalar(4, 1e-2)] if physics == "rb" else []
    s = State(p, {"ns": abi.TH_NS, "mhd": abi.TH_MHD, "rb": abi.TH_RB}[physics])
    s.upload([p.to_dev(v) for v in F])
    if physics == "ns":
        s.step(1e-3, nu=5e-3, steps=2)
        o.rk4_ns(F, 5e-3, 1e-3, steps=2)
    elif physics == "mhd":
        s.step(1e-3, nu=5e-3, eta=4e-3, steps=2)
        o.rk4_mhd(F[:3], F[3:], 5e-3, 4e-3, 1e-3, steps=2)
    else:
        s.step(1e-3, Ra=1e4, Pr=1.0, steps=2)
        o.rk4_rb(F[:3], F[3], 1e4, 1.0, 1e-3, steps=2)
    m = max(np.abs(v).max() for v in F)
    for got, ref in zip(s.download(), F):
        assert np.abs(got.cpu().numpy() - ref).max() <= tol * m


@pytest.mark.parametrize("prec", ("fp64", "fp32"))
def test_short_boxes_in_an_ensemble_equal_single_boxes(ctx, prec):
    from tarang_amd import Ensemble, Plan, State
    shapes = [(64, 64, 64)] * 20 + [(32, 32, 32)] * 3
    V = {N: Oracle(N).ic_random(3, E0=0.5, kp=3.0) for N in set(shapes)}
    e = Ensemble(ctx, shapes, precision=prec)
    for b, N in enumerate(shapes):
        e.upload(b, [e.plan(b).to_dev(v) for v in V[N]])
    e.step(np.full(len(shapes), 1e-3), np.full(len(shapes), 5e-3), steps=2)
    for b in (0, 19, 20, 22):
        p = Plan(ctx, shapes[b], precision=prec)
        s = State(p)
        s.upload([p.to_dev(v) for v in V[shapes[b]]])
        s.step(1e-3, nu=5e-3, steps=2)
        for got, ref in zip(e.download(b), s.download()):
            assert np.array_equal(got.cpu().numpy(), ref.cpu().numpy())


# enough boxes for the x-forward with one tile of columns per workgroup, where one box takes the side-by-side one
@pytest.mark.parametrize("N,boxes", [((24, 128, 128), 8), ((32, 96, 128), 8), ((48, 96, 96), 7), ((64, 64, 64), 10),
                                     ((96, 96, 96), 3), ((96, 24, 48), 40), ((128, 64, 64), 4), ((16, 64, 64), 60)])
@pytest.mark.parametrize("prec", ("fp64", "fp32"))
def test_many_boxes_equal_one_box(ctx, N, boxes, prec):
    from tarang_amd import Ensemble, Plan, State
    print(N, boxes, prec, flush=True)
    V = Oracle(N).ic_random(3, E0=0.5, kp=3.0)
    e = Ensemble(ctx, [N] * boxes, precision=prec)
    for b in range(boxes):
        e.upload(b, [e.plan(b).to_dev(v * (1.0 if b < boxes - 1 else 0.5)) for v in V])
    e.step(np.full(boxes, 1e-3), np.full(boxes, 5e-3), steps=2)
    p = Plan(ctx, N, precision=prec)
    for b, f in ((0, 1.0), (boxes - 1, 0.5)):
        s = State(p)
        s.upload([p.to_dev(v * f) for v in V])
        s.step(1e-3, nu=5e-3, steps=2)
        for got, ref in zip(e.download(b), s.download()):
            assert np.array_equal(got.cpu().numpy(), ref.cpu().numpy())


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-5)])
def test_chained_rb_step_after_other_uses_of_the_state(ctx, prec, tol):
    """Short RB boxes step chained: what else uses the state's buffers between steps must not reach the next step, and
    the stage field stays readable."""
    from tarang_amd import Plan, State, abi
    N = (32, 24, 48)
    print(N, prec, flush=True)
    o = Oracle(N, basis="SCFT")
    p = Plan(ctx, N, basis="SCFT", precision=prec)
    F = o.ic_random(7, E0=0.5, kp=3.0) + [o.ic_random_scalar(4, 1e-2)]
    s = State(p, abi.TH_RB)
    s.upload([p.to_dev(v) for v in F])

    def step_and_check(what):
        s.step(1e-3, Ra=1e4, Pr=1.0, steps=1)
        o.rk4_rb(F[:3], F[3], 1e4, 1.0, 1e-3, steps=1)
        m = max(np.abs(v).max() for v in F)
        for got, ref in zip(s.download(), F):
            assert np.abs(got.cpu().numpy() - ref).max() <= tol * m, what

    step_and_check("start")
    step_and_check("again")
    assert all(np.isfinite(b.cpu().numpy()).all() for b in s.download_buffer(1))
    for stage in (1, 2, 3, 4):
        s.profile_passes(1e-3, Ra=1e4, Pr=1.0, stage=stage, nrep=2)
    step_and_check("profile")
    s.tune(1e-3, Ra=1e4, Pr=1.0, nrep=1)
    step_and_check("tune")
    F = [0.5 * v for v in F]
    s.upload([p.to_dev(v) for v in F])
    step_and_check("upload")


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-5)])
@pytest.mark.parametrize("N", [(16, 32, 24), (24, 64, 64), (32, 16, 128)])
def test_short_lines_keep_the_last_stage_field(ctx, N, prec, tol):
    """The input of the last RK4 stage after a step, from the oracle's step with a force of zero supply; NS, and MHD's
    U with B = 0."""
    from tarang_amd import Plan, State, abi
    print(N, prec, flush=True)
    o = Oracle(N)
    p = Plan(ctx, N, precision=prec)
    V = o.ic_random(8, E0=0.5, kp=3.0)
    d = [p.to_dev(v) for v in V]
    last = o.zeros(3)
    o.step_ns_forced(V, 0.01, 1e-3, 1, 1.0, 2.0, 0.0, 0.0, steps=2, last_stage=last)
    m = max(np.abs(v).max() for v in last)
    for physics in (abi.TH_NS, abi.TH_MHD):
        s = State(p, physics)
        s.upload(d + [p.to_dev(np.zeros_like(v)) for v in V] * (physics == abi.TH_MHD))
        s.step(1e-3, nu=0.01, eta=0.01, steps=2)
        for got, ref in zip(s.download_buffer(1)[:3], last):
            assert np.abs(got.cpu().numpy() - ref).max() <= tol * m
