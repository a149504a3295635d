"""Writes tests/golden/split_step.npz: the fields of one split-precision step from
seeded states.  The committed file is of the build before the role kernels (commit
ca2b3fd; the build of today is within 1.2e-15 of it).  Run on a GPU from the root of
the tree whose library is to be recorded:

    python3 <this file> <output .npz>

tests/test_gpu_split_golden.py compares the library with them.  Arrays only.
"""
import importlib
import os
import sys

import numpy as np

DIMS = [(9, 8, 1), (9, 8, 3)]
T0, DT, NSTEP = 0.5, 0.01, 3


def state(nx, ny, nz):
    """(q, e, p, u, up) of interior cells: flow, shear and anisotropy everywhere, so that
    every float term of the sources and fluxes counts.  Additions, products, quotients
    and square roots only: the same values on any host."""
    rng = np.random.default_rng(nx * ny * nz)
    n, t = nx * ny * nz, T0 + NSTEP * DT
    e = 20.0 * (1.0 + 0.2 * rng.uniform(-1, 1, n))
    pl = e * rng.uniform(0.2, 0.4, n)

    def velocity():
        ux, uy, un = 0.4 + 0.1 * rng.uniform(-1, 1, n), 0.1 * rng.uniform(-1, 1, n) - 0.3, 0.2 * rng.uniform(-1, 1, n)
        return np.stack([np.sqrt(1 + ux * ux + uy * uy + t * t * un * un), ux, uy, un])

    u, up = velocity(), velocity()
    pi = 0.02 * e * rng.uniform(-1, 1, (10, n))
    pt = 0.5 * (e - pl)
    f = np.sqrt(1 + u[1] * u[1] + u[2] * u[2])
    z = np.stack([t * u[3] / f, 0 * f, 0 * f, u[0] / t / f])
    g = np.array([1.0, 0.0, 0.0, 0.0])
    q = np.zeros((15, n))
    for m in range(4):
        q[m] = (e + pt) * u[0] * u[m] - pt * g[m] + (pl - pt) * z[0] * z[m] + pi[m]
    q[4] = pl
    q[5:] = pi
    return q, e, e / 3, u, up


def step(V, dims):
    """The fields after the step, stacked: q, e, u."""
    c = V.Vah(*dims, 0.1, 0.12, 0.3, DT, 0.2, T0, precision=1)
    c.set_state(NSTEP, *state(*dims))
    c.step(1)
    c.synchronize()
    s = c.state()
    c.close()
    return np.vstack([s["q"], s["e"][None], s["u"]])


if __name__ == "__main__":
    sys.path.insert(0, os.getcwd())
    V = importlib.import_module("gpu-vah_amd")
    np.savez_compressed(sys.argv[1], **{"x".join(map(str, d)): step(V, d) for d in DIMS})
