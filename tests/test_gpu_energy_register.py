"""GPU parity of the energy pass on the register FFT against the oracle: powers
of two from 512 to 4096, and Bluestein lengths at both ends of the convolution
sizes, with ensembles that fill part of a workgroup, and several rounds of it.

Tolerance: each transform is good to a few 1e-16 of the spectrum's norm, twice
that through Bluestein's two transforms, so mode energies agree to 1e-13 of the
largest.
"""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,copies", [(512, 1), (512, 4100), (1024, 3), (1024, 3100), (2048, 5), (4096, 2),
                                      (4096, 800), (23, 70), (61, 5), (64 + 3, 1), (129 * 2 - 1, 33), (262, 3),
                                      (509, 9), (514, 2), (1009, 800), (1027, 3), (2047, 2), (2059, 2), (4093, 3)])
@pytest.mark.parametrize("model", ["FPUT", "DNLS"])
def test_energies(gpu, model, n, copies):
    N = gpu
    s0 = np.random.default_rng(n + copies).normal(size=(copies, n, 2))
    with N.Ensemble(N.MODELS[model], n, copies, 0.01, beta=1.0) as ens:
        ens.upload(s0)
        e, _ = ens.linenergies()
        raw = ens.linenergies_raw()
    if model == "DNLS":
        want = O.linenergies_dnls(s0)
        norm = 1.0 / n / copies
    else:
        want = O.linenergies_real(s0, O.dispersion_real(n, 0.0))
        norm = 0.5 / copies / n
    assert np.abs(raw - want).max() <= 1e-13 * want.max()
    ref = O.calc_linenergies(want, norm, True)
    assert np.abs(e - ref).max() <= 1e-13 * ref.max()


@pytest.mark.parametrize("n", [2, 3, 4, 5, 6, 7, 9, 10, 12, 14, 15, 18, 20, 21, 24, 25, 27, 28, 30, 35, 48, 49, 60, 96, 100,
                               105, 126, 225, 343, 360, 500, 648, 1000, 1225, 1536, 2401, 3000, 4050, 5000, 7000, 8000])
@pytest.mark.parametrize("model", ["FPUT", "DNLS"])
def test_smooth_lengths(gpu, model, n):
    """The in-place sweeps: one chain, and an ensemble with a partly filled
    last round of a workgroup."""
    for copies in (1, max(3, 40001 // n)):
        test_energies(gpu, model, n, copies)


@pytest.mark.parametrize("n,copies", [(8192, 3), (8192, 700), (9000, 2), (10000, 1), (15625, 1), (16384, 300),
                                      (16807, 1), (20000, 1), (32768, 2), (65536, 140)])
@pytest.mark.parametrize("model", ["FPUT", "DNLS"])
def test_rows_of_long_chains(gpu, model, n, copies):
    """Even and odd numbers of rows, several chains to a workgroup, the longest."""
    test_energies(gpu, model, n, copies)
