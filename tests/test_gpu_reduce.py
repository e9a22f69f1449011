"""GPU parity of the mirror-group sums (energies, Sn, shell spectra, helicity, entropy, shell products) on fields
with no symmetry at all, every stored mode nonzero, against the FP64 oracle.

Each sum of n terms accumulates an error of at most n ulp of the sum of |terms|, in practice a few: the tolerance
is 1e-13 of the sum of |terms| (of the largest bin for spectra); mode counts are compared exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from pyoracle import Oracle  # noqa: E402

TOL = 1e-13


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available(), "GPU test run without a GPU"
    from tarang_amd import Context
    return Context(0)


# smallest lengths (every mode its own mirror or on a Nyquist plane), odd half-lengths, more modes than one launch
# has threads for, and a box whose bins exceed the four-copy table
@pytest.mark.parametrize("N,kf", [((4, 4, 4), (1.0, 1.0, 1.0)), ((4, 6, 8), (1.0, 1.0, 1.0)), ((12, 4, 12), (1.0, 0.5, 2.0)),
                                  ((24, 16, 12), (1.0, 1.0, 1.0)), ((128, 192, 96), (1.0, 1.0, 1.0)),
                                  ((8, 8, 8), (150.0, 170.0, 190.0))])
@pytest.mark.parametrize("basis,dealias", [("FOUR", True), ("FOUR", False), ("SCFT", True)])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_sums_over_mirror_groups(ctx, N, kf, basis, dealias, prec):
    from tarang_amd import Plan
    print(N, kf, basis, dealias, prec, flush=True)
    o = Oracle(N, kfactor=kf, basis=basis, dealias=dealias)
    p = Plan(ctx, N, kfactor=kf, basis=basis, precision=prec, dealias=dealias)
    rng = np.random.default_rng(3)
    V = [rng.standard_normal(o.shape) + 1j * rng.standard_normal(o.shape) for _ in range(6)]
    d = [p.to_dev(v) for v in V]
    if prec == "fp32":                      # the oracle sees the same rounded inputs
        V = [np.ascontiguousarray(x.cpu().numpy().astype(np.complex128)) for x in d]
    U, W = V[:3], V[3:]
    size = sum(o.energy(a) for a in U + W)

    def near(a, b, scale):
        assert np.abs(np.asarray(a) - np.asarray(b)).max() <= TOL * scale, (a, b)
    for a, da, w, dw in zip(U, d[:3], W, d[3:]):
        near(p.energy(da), o.energy(a), size)
        near(p.energy(da, dw), o.energy(a, w), size)
        for n in (0, 2):
            near(p.Sn(da, n), o.Sn(a, n), 4 * abs(o.Sn(a, n)))
            Sg, cg = p.shell_spectrum(da, None, n)
            So, co = o.shell_spectrum(a, None, n)
            assert np.array_equal(cg, co)
            near(Sg, So, np.abs(So).max())
        near(p.shell_spectrum(da, dw)[0], o.shell_spectrum(a, w)[0], np.abs(o.shell_spectrum(a, None)[0]).max())
        near(p.entropy_scalar(da), o.entropy_scalar(a), abs(o.entropy_scalar(a)))
    near(p.entropy(d[:3]), o.entropy(U), abs(o.entropy(U)))
    kmax = max(o.kmag(N[0] // 2, N[1] // 2, N[2] // 2), 1.0)
    hg, ho = p.helicity(d[:3]), o.helicity(U)
    near(hg[[0, 3]], np.asarray(ho)[[0, 3]], 4 * kmax * size)
    near(hg[2], ho[2], 4 * kmax ** 3 * size)
    near(p.shell_helicity(d[:3]), o.shell_helicity(U), 4 * kmax * size)
    radii = np.array([0.0, 1.0, 2.5, 4.0, 1e4])
    near(p.shell_mult_all(d[:3], d[3:], radii), o.shell_mult_all(U, W, radii), 4 * size)
    near(p.shell_mult_single(d[:3], d[3:], 1.0, 3.0), sum(o.shell_mult_single(a, w, 1.0, 3.0) for a, w in zip(U, W)), 4 * size)
