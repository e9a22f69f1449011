"""Forced FP32 steps against stored results.

The supply of a band mode is divided by 2 E and 1 - sk^2, so the force of a weak or nearly helical mode amplifies the last
bits of the FP32 fields: the inputs below are such ones, on which any other rounding in the passes (another radix
schedule, another fused product, the short-box kernels) moves the result by far more than the step's own accuracy.
tests/golden/forced_fp32.npz holds the band's modes after the steps, as the passes of forced FP32 states gave them when
they were the only ones.

Tolerance: the same passes give the same bits; the force itself is evaluated in FP64 by kernels whose sums may be ordered
otherwise, which can move single FP32 values by their last bit, 6e-8: 1e-6 leaves room for the amplification of such a
flip that the unforced part of the accuracy has (5e-8 of the largest value), and every stored input moves by 5e-6 or more
under another set of roundings."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FORCE = dict(proc=1, inner=1.5, outer=3.5, p3=0.3, p4=0.1)
STEPS, DT, NU = 4, 0.02, 5e-3
GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "forced_fp32.npz")


def waves(N):
    k = [np.fft.fftfreq(N[0], 1.0 / N[0]), np.fft.fftfreq(N[1], 1.0 / N[1]), np.arange(N[2] // 2 + 1.0)]
    return k[0][:, None, None], k[1][None, :, None], k[2][None, None, :]


def field(N, seed):
    """Three random solenoidal components on |k_i| < N_i / 3 with energy 1/2, real in space, in complex64."""
    rng = np.random.default_rng(seed)
    kx, ky, kz = waves(N)
    k2 = kx * kx + ky * ky + kz * kz
    keep = (abs(kx) < N[0] // 3) & (abs(ky) < min(N[1] // 3, N[1] - 2 * (N[1] // 3) - 1)) & (kz < N[2] // 3)
    amp = np.where(keep & (k2 > 0), 1.0 / (1.0 + k2 * k2 / 64.0), 0.0)
    out = []
    for _ in range(3):
        a = (rng.standard_normal(amp.shape) + 1j * rng.standard_normal(amp.shape)) * amp
        m = np.roll(a[::-1, ::-1, 0], (1, 1), (0, 1))
        a[:, :, 0] = 0.5 * (a[:, :, 0] + m.conj())
        out.append(a)
    d = (kx * out[0] + ky * out[1] + kz * out[2]) / np.where(k2 > 0, k2, 1.0)
    out = [a - k * d for a, k in zip(out, (kx, ky, kz))]
    e = sum((a.real ** 2 + a.imag ** 2).sum() for a in out)
    return [(a * np.sqrt(0.5 / e)).astype(np.complex64) for a in out]


def band(N):
    kx, ky, kz = waves(N)
    k = np.sqrt(kx * kx + ky * ky + kz * kz)
    return (k > FORCE["inner"]) & (k <= FORCE["outer"])


def run(abi, ctx, N, seed):
    p = abi.Plan(ctx, N, precision="fp32")
    s = abi.State(p)
    s.upload([p.to_dev(v) for v in field(N, seed)])
    s.set_force(**FORCE)
    s.step(DT, nu=NU, steps=STEPS)
    return np.stack([a.cpu().numpy()[band(N)] for a in s.download()])


# chained steps on 2^a and 3 2^a lines, short and long ones, and lines of 32, which step unchained
CASES = [((32, 16, 16), 88), ((48, 16, 32), 184), ((64, 24, 16), 266), ((192, 16, 16), 161), ((256, 16, 24), 220)]


@pytest.mark.parametrize("N,seed", CASES)
def test_forced_fp32_step_keeps_its_results(N, seed):
    import torch
    assert torch.cuda.is_available(), "GPU test run without a GPU"
    from tarang_amd import Context, abi
    print(N, seed, flush=True)
    ref = np.load(GOLDEN)["%dx%dx%d_%d" % (*N, seed)]
    got = run(abi, Context(0), N, seed)
    assert np.linalg.norm(got - ref) <= 1e-6 * np.linalg.norm(ref)
