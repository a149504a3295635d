"""The stage kernels' tiles at their edges: lattices one cell short of a tile, one
tile, one cell over and odd remainders, each eta chunk the launch rule picks, and the
wide tiles, which long lattices of few columns reach (the rule counts workgroups)."""
import numpy as np
import pytest

from tests.parity import TOL_FP64, assert_parity, gaussian_ic, rest_frame, vah

pytestmark = pytest.mark.gpu

STEPS = 3


def run(V, oracle_mod, nx, ny, nz, precision, eta_chunk):
    e = gaussian_ic(nx, ny, nz, dz=0.3 if nz < 100 else 6.0 / nz, seed=nx + ny + nz, peak=60.0, tilt=0.2)
    # the vacuum tail of a long lattice stays out of the comparison
    e = np.maximum(e, 1.0)
    dz = 0.3
    g = V.Vah(nx, ny, nz, 0.1, 0.1, dz, 0.01, 0.2, 0.5, precision=precision, eta_chunk=eta_chunk)
    o = oracle_mod.Oracle(nx, ny, nz, 0.1, 0.1, dz, 0.01, 0.2, 0.5)
    for x in (g, o):
        x.set_primitives(e, *rest_frame(e.size), pl=e / 3)
        x.step(STEPS)
    g.synchronize()
    a, b, tau = g.state(), o.state(), o.time
    g.close()
    o.close()
    return a, b, tau


def check(a, b, tau, precision, label):
    if precision == 0:
        assert_parity(a, b, tau, TOL_FP64, label=label)
    else:  # float arithmetic in double storage: the split form's bound on e and u
        assert np.max(np.abs(a["e"] - b["e"]) / b["e"]) < 1e-4
        assert np.max(np.abs(a["u"] - b["u"]) / b["u"][0]) < 1e-4


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "split"])
@pytest.mark.parametrize("dims", [(7, 6, 1), (8, 7, 1), (9, 8, 1), (15, 13, 1), (17, 15, 1), (65, 1, 1), (1, 29, 1)])
def test_2d_tile_edges(oracle_mod, dims, precision):
    check(*run(vah(), oracle_mod, *dims, precision, 0), precision, str(dims))


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "split"])
@pytest.mark.parametrize("dims,eta_chunk", [((7, 6, 3), 1), ((8, 7, 2), 2), ((9, 8, 5), 2), ((15, 13, 7), 3),
                                            ((17, 15, 13), 6), ((9, 15, 6), 6), ((8, 8, 4), 0)])
def test_3d_tile_edges(oracle_mod, dims, eta_chunk, precision):
    check(*run(vah(), oracle_mod, *dims, precision, eta_chunk), precision, f"{dims} {eta_chunk}")


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "split"])
@pytest.mark.parametrize("dims,eta_chunk", [((17, 8, 1725), 0), ((16, 14, 3450), 0), ((15, 13, 3448), 6),
                                            ((33, 15, 766), 4)])
def test_wide_tile_edges(oracle_mod, dims, eta_chunk, precision):
    check(*run(vah(), oracle_mod, *dims, precision, eta_chunk), precision, f"{dims} {eta_chunk}")
