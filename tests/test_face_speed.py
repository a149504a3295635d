"""The closed-form face speed of the stage kernels (gpu-vah_amd/csrc/vah_face.h,
compiled for the host from the same header) against the oracle's Newton
iteration (EnergyMomentumTensor.cpp:30-72) from the same start: wherever the
closed form is taken, the iteration succeeds and gives the same speed."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from tests.test_oracle_math import conserved_from_primitives, p, random_primitives

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-vah_amd", "csrc")

SRC = r'''
#define __host__
#define __device__
#include FACE_H
// 1 when the closed form applies; v[0..2]: the speeds along x, y, eta
extern "C" int face(double t, const double *q, double u0, double *v) {
    const vah::FaceStart s = vah::face_start(u0 * u0);
    double M[4];
    for (int m = 0; m < 4; ++m) M[m] = q[m] - q[5 + m];
    const bool a = vah::face_speed<1>(t, M[0], M[1], M[2], M[3], q[4], s, v);
    const bool b = vah::face_speed<2>(t, M[0], M[1], M[2], M[3], q[4], s, v + 1);
    const bool c = vah::face_speed<3>(t, M[0], M[1], M[2], M[3], q[4], s, v + 2);
    return a == b && b == c ? (int)a : -1;
}
'''


@pytest.fixture(scope="module")
def face(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("face")
    (d / "f.cpp").write_text(SRC.replace("FACE_H", '"' + os.path.join(CSRC, "vah_face.h") + '"'))
    subprocess.run(["g++", "-O2", "-shared", "-fPIC", "-o", str(d / "f.so"), str(d / "f.cpp")], check=True)
    f = ctypes.CDLL(str(d / "f.so")).face
    dp = ctypes.POINTER(ctypes.c_double)
    f.argtypes = [ctypes.c_double, dp, ctypes.c_double, dp]
    return f


def _state(rng, t, kind):
    """(q, u0, physical): near starts, far starts, unphysical states, light-like flow."""
    if kind == 2:
        q = np.zeros(15)
        q[0] = 10 ** rng.uniform(-3, 2)
        q[1:4] = rng.normal(0, 1, 3) * q[0]
        q[3] /= t
        q[4] = q[0] * rng.uniform(-0.1, 1.0)
        q[5:15] = rng.normal(0, 0.1, 10) * q[0]
        return q, 10 ** rng.uniform(-4, 1.5), False
    e, pl, ut, ux, uy, un, pi = random_primitives(rng, t)
    s = 10 ** rng.uniform(0.5, 1.5) if kind == 3 else 1.0
    ux, uy = ux * s, uy * s
    ut = np.sqrt(1 + ux * ux + uy * uy + t * t * un * un)
    uT = np.hypot(ux, uy)
    return conserved_from_primitives(t, e, pl, ut, ux, uy, un, pi), \
        (10 ** rng.uniform(-6, 3) if kind == 1 else uT * rng.uniform(0.5, 1.5)), True


def test_closed_form_speed_is_where_the_newton_path_ends(oracle_mod, face):
    """20,000 states of four kinds.  Both the iteration's stopping rule
    (|du| <= 1e-7 u, quadratic: ~1e-14) and the conditioning of the root near
    light-like flow (gamma^2 ~ 1e3 times rounding) bound the agreement: 1e-11
    of the larger of v and the oracle's |u_T| / u^tau."""
    L = oracle_mod.lib()
    rng = np.random.default_rng(17)
    out, v = np.zeros(6), np.zeros(3)
    fired = physical = 0
    worst = 0.0
    for k in range(20000):
        t = rng.uniform(0.3, 5.0)
        q, u0, phys = _state(rng, t, k % 4)
        got = face(t, p(q), u0, p(v))
        assert got in (0, 1)
        # starts near the root of a physical state: the closed form must be taken
        physical += phys and k % 4 != 1
        fired += got and phys and k % 4 != 1
        if not got:
            continue
        assert L.orc_recover(t, p(q), 1.0, u0, p(out)) == 0, (k, t, u0)
        want = out[3:6] / out[2]
        scale = max(np.hypot(want[0], want[1]), 1e-12)
        worst = max(worst, *(abs(v[:2] - want[:2]) / scale), abs(v[2] - want[2]) / max(abs(want[2]), 1e-12))
    assert fired > 0.98 * physical, (fired, physical)
    assert worst < 1e-11, worst


@pytest.mark.parametrize("u0", [0.0, 1e-8, 0.3])
def test_state_at_rest(oracle_mod, face, u0):
    """A state exactly at rest gives v = 0 from any start it accepts; from a
    zero start it is accepted (the initial state of every event)."""
    q = conserved_from_primitives(0.5, 10.0, 3.0, 1.0, 0.0, 0.0, 0.0, np.zeros(10))
    v = np.ones(3)
    got = face(0.5, p(q), u0, p(v))
    assert got == 1 if u0 == 0.0 else got in (0, 1)
    if got:
        assert np.all(v == 0.0)


@pytest.mark.parametrize("break_", ["nan", "inf", "zero", "luminal"])
def test_broken_states_go_to_the_iteration(face, break_):
    q = conserved_from_primitives(0.5, 10.0, 3.0, 1.0, 0.0, 0.0, 0.0, np.zeros(10))
    if break_ == "nan":
        q[1] = np.nan
    elif break_ == "inf":
        q[0] = np.inf
    elif break_ == "zero":
        q[:] = 0.0
    else:
        q[3] = 1.0001 * (q[0] + q[4]) / 0.5
    assert face(0.5, p(q), 0.1, p(np.zeros(3))) == 0
