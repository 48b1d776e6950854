"""GPU parity of the DNLS register kernels of 32 to 2048 sites against the
oracle: every length, ensembles that leave chain slots of the last wavefront
empty, angles beyond the short sin/cos form.

Tolerance: the two transforms each round at a few ulp per pass, so a substep
moves a chain by about 1e-15 of its norm; 7 substeps x 30 steps growing
linearly stay below 1e-12.
"""
import numpy as np
import pytest

from oracle import oracle as O
from parity import chain_rel_err

pytestmark = pytest.mark.gpu


def check(N, n, copies, beta, sample=None):
    steps, dt = (30 if n < 8192 else 5, 0.01) if beta == 1.0 else (5, 0.02)
    s0 = N.ic_dnls(n, copies, max(1, n // 16), 1.0, 9) + 0.05 * np.random.default_rng(n).normal(size=(copies, n, 2))
    with N.Ensemble(N.DNLS, n, copies, dt, beta=beta) as ens:
        ens.upload(s0)
        ens.move(steps)
        got = ens.download()
    if sample is not None:
        got, s0 = got[sample], s0[sample]
    assert chain_rel_err(got, O.move_dnls(s0, steps, dt, beta)) <= 1e-12


@pytest.mark.parametrize("n", [32, 64, 128, 256, 512, 1024, 2048])
@pytest.mark.parametrize("copies", [1, 19])
@pytest.mark.parametrize("beta", [1.0, 60.0])
def test_register_lengths(gpu, n, copies, beta):
    check(gpu, n, copies, beta)


@pytest.mark.parametrize("n,copies", [(128, 8192), (256, 4097), (512, 6147), (1024, 3073), (2048, 1537), (4096, 5),
                                      (8192, 128), (16384, 129)])
def test_register_lengths_of_large_ensembles(gpu, n, copies):
    """The shapes with more values per thread, at the first sizes that take
    them; the first, some middle and the last chains."""
    check(gpu, n, copies, 1.0, [0, 1, copies // 2, copies - 2, copies - 1])


@pytest.mark.parametrize("n", [11, 17, 33, 67, 131, 262, 521, 1027, 2059])
@pytest.mark.parametrize("copies", [1, 19])
def test_bluestein_lengths(gpu, n, copies):
    """Lengths just above a power of two (the longest padding) and their
    neighbours: convolutions of 32 to 8192 points, each twice the transforms of
    test_register_lengths over fewer steps."""
    N = gpu
    steps = 20 if n < 600 else 3
    s0 = N.ic_dnls(n, copies, max(1, n // 16), 1.0, 9) + 0.05 * np.random.default_rng(n).normal(size=(copies, n, 2))
    with N.Ensemble(N.DNLS, n, copies, 0.01, beta=1.0) as ens:
        ens.upload(s0)
        ens.move(steps)
        got = ens.download()
    assert chain_rel_err(got, O.move_dnls(s0, steps, 0.01, 1.0)) <= 1e-12


@pytest.mark.parametrize("n,copies", [(61, 8193), (127, 4097), (251, 6145), (509, 3073), (1021, 1537)])
def test_bluestein_lengths_of_large_ensembles(gpu, n, copies):
    """The convolution shapes with more values per thread (sizes just below a
    power of two)."""
    N = gpu
    steps, at = 3, [0, 1, copies // 2, copies - 2, copies - 1]
    s0 = N.ic_dnls(n, copies, max(1, n // 16), 1.0, 9)
    with N.Ensemble(N.DNLS, n, copies, 0.01, beta=1.0) as ens:
        ens.upload(s0)
        ens.move(steps)
        got = ens.download()
    assert chain_rel_err(got[at], O.move_dnls(s0[at], steps, 0.01, 1.0)) <= 1e-12


@pytest.mark.parametrize("n", [2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 14, 15, 16, 18, 20, 21, 24, 25, 27, 28, 30, 35, 45, 48, 49,
                               60, 96, 98, 100, 105, 120, 126, 150, 196, 210, 225, 243, 343, 350, 500, 648, 980, 1000,
                               1225, 1536, 2187, 2401, 3000, 4050, 5000, 6561, 7000, 8000])
def test_smooth_lengths(gpu, n):
    """Every radix in the outer, middle and inner sweep (two to five passes),
    one chain and an ensemble that ends inside a workgroup."""
    N = gpu
    steps = 20 if n < 700 else 2
    for copies in (1, 700 if n < 130 else 19 if n < 700 else 2):
        s0 = N.ic_dnls(n, copies, max(1, n // 16), 1.0, 9) + 0.05 * np.random.default_rng(n).normal(size=(copies, n, 2))
        with N.Ensemble(N.DNLS, n, copies, 0.01, beta=1.0) as ens:
            ens.upload(s0)
            ens.move(steps)
            got = ens.download()
        at = [0, copies // 2, copies - 1]
        assert chain_rel_err(got[at], O.move_dnls(s0[at], steps, 0.01, 1.0)) <= 1e-12


@pytest.mark.parametrize("n,copies", [(96, 9000), (100, 5001), (360, 3001), (1000, 1025), (3000, 600)])
def test_smooth_lengths_of_large_ensembles(gpu, n, copies):
    """Several chains per workgroup, the last workgroup partly filled."""
    N = gpu
    steps, at = 2, [0, 1, 2, 3, copies // 2, copies - 2, copies - 1]
    s0 = N.ic_dnls(n, copies, max(1, n // 16), 1.0, 9)
    with N.Ensemble(N.DNLS, n, copies, 0.01, beta=1.0) as ens:
        ens.upload(s0)
        ens.move(steps)
        got = ens.download()
    assert chain_rel_err(got[at], O.move_dnls(s0[at], steps, 0.01, 1.0)) <= 1e-12
