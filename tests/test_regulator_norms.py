"""The regulator's norms (gpu-vah_amd/csrc/vah_div.h: root_of and the quotient by a
root, which vah_source.h takes sqrt(|pi:pi|), its inverse and rho from) keep the
rounding of the square roots and divisions of the reference's sequence
(FullyDiscreteKurganovTadmorScheme.cpp:540-665), from seeds off by up to 2^-22."""
import ctypes
import shutil

import numpy as np
import pytest

from tests.test_seed_error import build

SRC = r'''
#define __host__
#define __device__
#include FACE_H
extern "C" void norms(long n, const double *pipi2, const double *s2, double *spipi, double *ispipi, double *rho) {
    for (long k = 0; k < n; ++k) {
        const vah::Root r = vah::root_of(pipi2[k]);
        spipi[k] = r.root, ispipi[k] = r.inverse;
        rho[k] = vah::quotient(r.root, vah::root_of(s2[k]));
    }
}
'''


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("decades", [3, 270])
def test_norms_round_as_the_library_sequence(tmp_path, decades):
    """Bit for bit against sqrt and division; the inverse may miss by one unit where the
    root's mantissa is nearly all ones (fewer than one case in 1e5)."""
    n = 500000
    rng = np.random.default_rng(decades)
    pipi2 = rng.uniform(1, 10, n) * 10.0 ** rng.uniform(-decades, decades, n)
    s2 = pipi2 * rng.uniform(1, 10, n) * 10.0 ** rng.uniform(-2, 8, n) if decades < 10 else \
        rng.uniform(1, 10, n) * 10.0 ** rng.uniform(-decades, decades, n)
    got = [np.zeros(n) for _ in range(3)]
    f = ctypes.CDLL(build(tmp_path, SRC)).norms
    f(ctypes.c_long(n), *(x.ctypes.data_as(ctypes.c_void_p) for x in (pipi2, s2, *got)))
    want = [np.sqrt(pipi2), 1.0 / np.sqrt(pipi2), np.sqrt(pipi2) / np.sqrt(s2)]
    for a, b, name in zip(got, want, ("spipi", "ispipi", "rho")):
        off = a.view(np.int64) != b.view(np.int64)
        assert off.sum() <= (0 if name == "spipi" else n // 100000), (name, off.sum())
        assert np.all(np.abs(a.view(np.int64) - b.view(np.int64)) <= 1), name
