"""The range of the closed forms of the stage kernels (gpu-vah_amd/csrc/vah_face.h,
compiled for the host from the same header).  The equations are homogeneous: a state
times s has the same velocity and face speeds, and s times its e.  A scaled state
either gives exactly that or goes to the iteration, also where the squares of the
root overflow or underflow."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from tests.test_oracle_math import conserved_from_primitives, p

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-vah_amd", "csrc")

SRC = r'''
#define __host__
#define __device__
#include FACE_H
// bit 0: the cell's closed form applies, bit 1: the faces'
// v: e, u^tau, u^x, u^y, u^eta, and the speeds along x, y, eta
extern "C" int both(double t, const double *q, double u0, double *v) {
    const vah::FaceStart s = vah::face_start(u0 * u0);
    double M[4];
    for (int m = 0; m < 4; ++m) M[m] = q[m] - q[5 + m];
    vah::CellRoot c;
    const bool cell = vah::cell_root(t, M[0], M[1], M[2], M[3], q[4], s, &c);
    v[0] = c.e, v[1] = c.ut, v[2] = c.ux, v[3] = c.uy, v[4] = c.un;
    const bool x = vah::face_speed<1>(t, M[0], M[1], M[2], M[3], q[4], s, v + 5);
    const bool y = vah::face_speed<2>(t, M[0], M[1], M[2], M[3], q[4], s, v + 6);
    const bool n = vah::face_speed<3>(t, M[0], M[1], M[2], M[3], q[4], s, v + 7);
    return (int)cell + 2 * (x && y && n);
}
'''


@pytest.fixture(scope="module")
def both(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("range")
    (d / "r.cpp").write_text(SRC.replace("FACE_H", '"' + os.path.join(CSRC, "vah_face.h") + '"'))
    subprocess.run(["g++", "-O2", "-shared", "-fPIC", "-o", str(d / "r.so"), str(d / "r.cpp")], check=True)
    f = ctypes.CDLL(str(d / "r.so")).both
    dp = ctypes.POINTER(ctypes.c_double)
    f.argtypes = [ctypes.c_double, dp, ctypes.c_double, dp]
    return f


@pytest.mark.parametrize("uT", [0.0, 1e-3, 0.5, 1.5, 3.0, 20.0])
def test_a_scaled_state_scales_or_goes_to_the_iteration(both, uT):
    """Powers of two from 2^-1000 to 2^1020.  They only shift exponents, so the
    agreement is to rounding (16 eps (u^tau)^2, the conditioning of the root)."""
    t, ux, uy, un = 0.5, 0.8 * uT, -0.6 * uT, 0.3
    ut = np.sqrt(1 + ux * ux + uy * uy + t * t * un * un)
    q = conserved_from_primitives(t, 1.0, 0.3, ut, ux, uy, un, np.zeros(10))
    base, v = np.zeros(8), np.zeros(8)
    assert both(t, p(q), uT, p(base)) == 3
    taken = 0
    for k in range(-1000, 1021):
        s = 2.0 ** k
        with np.errstate(over="ignore"):
            got = both(t, p(q * s), uT, p(v))
        taken += got == 3
        err = np.abs(v / np.r_[s, np.ones(7)] - base)
        bound = 16 * 2.3e-16 * ut ** 2 * np.maximum(np.abs(base), [q[0], 0, uT, uT, 0, uT / ut, uT / ut, 0])
        if got & 1:
            assert np.all(err[:5] <= bound[:5]), (k, v, base)
        if got & 2:
            assert np.all(err[5:] <= bound[5:]), (k, v, base)
    # the closed form is what runs: 280 decades, at rest the 149 below 1e9 (above, the
    # floor of the square root fails the first-update test and the iteration runs)
    assert taken > (480 if uT == 0.0 else 800)
