"""The launch geometry of the single-lattice stage kernels (gpu-vah_amd/csrc/
vah_geometry.h, compiled for the host): it covers every lattice, and the lattices of
the GPU tests take the tile shape and the chunks that these tests are about."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from tests import test_gpu_tiles
from tests.parity import gaussian_ic, rest_frame, vah
from tests.test_gpu_batch import admit, worst
from tests.test_gpu_tiles import check, run

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-vah_amd", "csrc")

SRC = r'''
#include GEOMETRY_H
extern "C" void geometry(int nx, int ny, int nz, int shared, int eta_chunk, int *o) {
    const vah::Geometry g = vah::launch_geometry(nx, ny, nz, shared, eta_chunk);
    o[0] = g.tiles_x, o[1] = g.tiles_y, o[2] = g.zchunks, o[3] = g.kz, o[4] = g.nblocks, o[5] = g.grid, o[6] = g.wide;
}
'''

# nz just under and over the rules' edges, the last chunk of six planes holding one:
# (lattice, tiles of 16 x 7 or 8 x 7, kz)
CHOSEN = [((17, 8, 1725), True, 3), ((17, 8, 1722), False, 3), ((17, 8, 3073), True, 6), ((17, 8, 3066), True, 3),
          ((17, 8, 766), False, 3), ((17, 8, 765), False, 2), ((17, 8, 511), False, 2), ((17, 8, 510), False, 1),
          ((611, 587, 1), False, 1), ((785, 1253, 1), False, 1), ((785, 1254, 1), True, 1),
          ((767, 9000, 1), False, 1), ((768, 1310, 1), True, 1), ((1001, 1001, 1), True, 1)]


@pytest.fixture(scope="module")
def geometry(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("geometry")
    (d / "g.cpp").write_text(SRC.replace("GEOMETRY_H", '"' + os.path.join(CSRC, "vah_geometry.h") + '"'))
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", str(d / "g.so"), str(d / "g.cpp")], check=True)
    f = ctypes.CDLL(str(d / "g.so")).geometry

    def call(dims, shared=True, eta_chunk=0):
        o = (ctypes.c_int * 7)()
        f(*dims, int(shared), eta_chunk, o)
        return dict(zip(("tiles_x", "tiles_y", "zchunks", "kz", "nblocks", "grid", "wide"), o))

    return call


def test_geometry_covers_the_lattice(geometry):
    rng = np.random.default_rng(4)
    for k in range(4000):
        dims = tuple(int(10 ** rng.uniform(0, top)) for top in (2.8, 2.8, 2.2))
        dims = dims[:2] + (1,) if k % 4 == 0 else dims
        shared, chunk = k % 3 != 0, int(rng.integers(0, 257)) if k % 2 else 0
        g = geometry(dims, shared, chunk)
        tx, ty = (16, 16) if not shared else (16 if g["wide"] else 8, 7)
        tiles = g["tiles_x"] * g["tiles_y"]
        assert 0 <= g["tiles_x"] * tx - dims[0] < tx and 0 <= g["tiles_y"] * ty - dims[1] < ty
        assert 1 <= g["kz"] <= dims[2] and 0 <= g["zchunks"] * g["kz"] - dims[2] < g["kz"]
        assert g["kz"] == min(chunk, dims[2]) or chunk == 0
        assert g["nblocks"] == tiles * g["zchunks"] and g["grid"] == g["zchunks"] * 8 * -(-tiles // 8)
        assert not g["wide"] or shared


def test_chosen_tiles_and_chunks(geometry):
    for dims, wide, kz in CHOSEN:
        g = geometry(dims)
        assert (bool(g["wide"]), g["kz"]) == (wide, kz), (dims, g)
        assert geometry(dims, shared=False)["kz"] == 1


def test_gpu_tile_tests_take_the_tiles_they_name(geometry):
    def cases(test):
        return next(m.args[1] for m in test.pytestmark if m.args and m.args[0] == "dims,eta_chunk")

    for dims, chunk in cases(test_gpu_tiles.test_wide_tile_edges):
        assert geometry(dims, eta_chunk=chunk)["wide"], dims
    for dims, chunk in cases(test_gpu_tiles.test_3d_tile_edges):
        assert not geometry(dims, eta_chunk=chunk)["wide"], dims


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "split"])
@pytest.mark.parametrize("dims", [(17, 8, 3073), (17, 8, 765), (17, 8, 766)])
def test_automatic_chunks(oracle_mod, dims, precision):
    """The chunks that the rule picks, with a last one of a single plane or two."""
    check(*run(vah(), oracle_mod, *dims, precision, 0), precision, str(dims))


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "split"])
@pytest.mark.parametrize("dims", [(785, 1254, 1), (799, 1261, 1), (768, 1310, 1)])
def test_wide_tiles_in_two_dimensions(geometry, dims, precision):
    """One cell over, on and under 16 and 7, against a batch of the one event in 8 x 7
    tiles (1e-12, as every event of a batch; split 1e-4 in e and u).  Not against the
    oracle: among a million lumpy cells some take another branch of the scheme there, by
    1.7e-10, in 8 x 7 tiles and in the kernels before the roles just the same."""
    assert geometry(dims)["wide"]
    V = vah()
    nx, ny, nz = dims
    e = np.maximum(gaussian_ic(nx, ny, nz, dz=0.3, seed=nx + ny + nz, peak=60.0, tilt=0.2), 1.0)
    g = V.Vah(nx, ny, nz, 0.1, 0.1, 0.3, 0.01, 0.2, 0.5, precision=precision)
    g.set_primitives(e, *rest_frame(e.size), pl=e / 3)
    g.step(3)
    g.synchronize()
    B = V.Batch(budget_bytes=V.batch_event_bytes(*dims) + (1 << 20), max_events=1, freezeout_T_GeV=0.0, variant=4,
                precision=precision)
    slot = admit(B, dict(nx=nx, ny=ny, nz=nz, dx=0.1, dy=0.1, dz=0.3, dt=0.01, t0=0.5, etabar=0.2, e=e))
    B.step(3)
    a, b, tau = g.state(), B.state(slot), B.poll()[0]["tau"]
    g.close()
    B.close()
    if precision == 0:
        assert worst(a, b, tau) <= 1e-12
    else:
        check(a, b, tau, precision, str(dims))


@pytest.mark.gpu
def test_per_cell_chunk():
    """The per-cell kernels' chunk of one plane computes what any chunk does."""
    V = vah()
    nx, ny, nz = 17, 18, 5
    e = np.maximum(gaussian_ic(nx, ny, nz, dz=0.3, seed=5, peak=60.0), 1.0)
    got = []
    for chunk in (0, 1, 3, 5):
        g = V.Vah(nx, ny, nz, 0.1, 0.1, 0.3, 0.01, 0.2, 0.5, flux_mode=V.FLUX_PER_CELL, eta_chunk=chunk)
        g.set_primitives(e, *rest_frame(e.size), pl=e / 3)
        g.step(3)
        g.synchronize()
        got.append(g.state())
        g.close()
    for s in got[1:]:
        assert all(np.array_equal(s[k], got[0][k]) for k in ("q", "e", "p", "u", "up"))
