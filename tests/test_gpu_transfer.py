"""Energy transfer with several giver shells in one launch (th_flux_shell_tr, th_flux_mhd_fused): every giver's row
equals that of a call with this giver alone, which runs in the state's own buffers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available(), "GPU test run without a GPU"
    from tarang_amd import Context
    return Context(0)


def state(ctx, N, prec, physics, seed):
    """Random real fields over the kept modes, |u(K)| ~ 1 / (1 + K^2)."""
    import torch
    from tarang_amd import Plan, State
    p = Plan(ctx, N, precision=prec)
    s = State(p, physics)
    gen = torch.Generator().manual_seed(seed)
    f = [torch.fft.fftfreq(n, 1.0 / n).abs() for n in N[:2]] + [torch.arange(N[2] // 2 + 1).double()]
    K2 = f[0][:, None, None] ** 2 + f[1][None, :, None] ** 2 + f[2][None, None, :] ** 2
    keep = (f[0] <= N[0] // 3)[:, None, None] & (f[1] <= N[1] // 3)[None, :, None] & (f[2] <= N[2] // 3)[None, None, :]
    out = []
    for _ in range(s.ncomp):
        u = torch.fft.rfftn(torch.randn(N, generator=gen, dtype=torch.float64)) / np.prod(N)
        out.append(p.to_dev((u * keep / (1.0 + K2)).numpy()))
    s.upload(out)
    return s


# planes of 16 to 64 points in one launch and not, more givers than one launch takes (64^3 FP64: 10), odd remainders,
# the numbers of shells at which the bins have fewer copies
SIZES = [((16, 16, 16), 5), ((24, 48, 32), 11), ((64, 64, 64), 21), ((32, 96, 96), 9), ((48, 128, 24), 7),
         ((32, 24, 32), 70), ((32, 24, 32), 140)]


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-11), ("fp32", 2e-5)])
@pytest.mark.parametrize("N,nsh", SIZES)
def test_givers_together_and_alone(ctx, N, nsh, prec, tol):
    print(f"transfer {prec} N={N} nsh={nsh}", flush=True)
    s = state(ctx, N, prec, 0, 7)
    radii = np.concatenate([np.arange(nsh, dtype=float) * min(1.25, 20.0 / nsh), [1e4]])
    Pi, T = s.flux_shell_tr(radii)
    again = s.flux_shell_tr(radii)
    scale = np.abs(T).max()
    assert np.abs(T - again[1]).max() <= tol * scale and np.isfinite(Pi).all()
    for n in range(1, nsh):
        _, t = s.flux_shell_tr(np.array([radii[n - 1], radii[n], 1e4]))
        assert abs(t[1, 1] - T[n, n]) <= tol * scale, n
        assert abs(t[1, 2] - T[n, n + 1:].sum()) <= tol * scale, n


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-11), ("fp32", 2e-5)])
def test_mhd_pipelines_share_the_workspace(ctx, prec, tol):
    """Two receivers, four pipelines with another helper or giver each, and another number of givers."""
    from tarang_amd import abi
    for N in ((32, 24, 48), (32, 96, 64)):
        print(f"mhd flux {prec} N={N}", flush=True)
        s = state(ctx, N, prec, abi.TH_MHD, 11)
        radii = np.concatenate([np.arange(8, dtype=float), [1e4]])
        got = s.flux_mhd(radii)
        for i in (1, 4, 7):       # out- and in-sphere rows of sphere i from its one giver (0, R_i]
            one = s.flux_mhd(np.array([0.0, radii[i], 1e4]))
            sel = [0, 1, 2, 3, 4, 5, 7, 8]
            assert np.abs(got[sel, i] - one[sel, 1]).max() <= tol * np.abs(got).max(), (N, i)
