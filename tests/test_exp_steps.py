"""exp2_256_tab (nlchains_amd/csrc/nlc_exp.hpp, the Toda kernels' form on table
steps), compiled on the host from the same header: the bits of exp2_128_tab on
half the argument where that one's reduction is exact, saturation beyond."""
import ctypes
import subprocess
from pathlib import Path

import numpy as np
import pytest

HEADER = Path(__file__).resolve().parents[1] / "nlchains_amd" / "csrc" / "nlc_exp.hpp"
WRAPPER = r"""
#define NLC_EXP_QUAL inline
#define NLC_EXP_HOST 1
#include "nlc_exp.hpp"
static const double tab[nlc::kExpTabSize] = NLC_EXP2_TABLE;
extern "C" void steps(const double *x, double *out, long n) {
	for (long i = 0; i < n; ++i) out[i] = nlc::exp2_256_tab(x[i], tab);
}
extern "C" void halves(const double *x, double *out, long n) {
	for (long i = 0; i < n; ++i) out[i] = nlc::exp2_128_tab(x[i] / 2, tab);
}
"""


@pytest.fixture(scope="module")
def forms(tmp_path_factory):
    d = tmp_path_factory.mktemp("exp256")
    (d / "w.cpp").write_text(WRAPPER)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", f"-I{HEADER.parent}",
                    str(d / "w.cpp"), "-o", str(d / "libw.so")], check=True)
    lib = ctypes.CDLL(str(d / "libw.so"))

    def call(fn, x):
        x = np.ascontiguousarray(x, dtype=np.float64)
        out = np.empty_like(x)
        fn(x.ctypes.data_as(ctypes.c_void_p), out.ctypes.data_as(ctypes.c_void_p), ctypes.c_long(x.size))
        return out
    return lambda x: (call(lib.steps, x), call(lib.halves, x))


def test_same_bits(forms):
    rng = np.random.default_rng(2)
    k = np.arange(-3000, 3000) / 4  # table points, their midpoints (ties) and quarters
    for x in (rng.uniform(-400, 400, 20000), rng.uniform(-3e5, 3e5, 20000), rng.uniform(-1e-4, 1e-4, 2000), k,
              np.nextafter(k, np.inf), np.nextafter(k, -np.inf), 2.0 ** rng.uniform(20, 50, 2000)):
        a, b = forms(x)
        assert np.array_equal(a, b)


def test_saturation(forms):
    x = 10.0 ** np.random.default_rng(3).uniform(6, 300, 4000)
    assert np.all(forms(x)[0] == np.inf) and np.all(forms(-x)[0] == 0.0)
    assert np.isnan(forms(np.array([np.nan, np.inf, -np.inf]))[0]).all()
