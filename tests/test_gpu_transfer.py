"""States to the device and back: every value returns as it was given, through
one chunk, several, chunks of one row longer than a transfer slot, fields with a
gap behind them, and sizes that several host threads share."""
import numpy as np
import pytest

from tests.test_gpu_batch import admit, vah

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (1, 9, 1), (33, 1, 1), (7, 5, 2), (41, 37, 1), (60, 60, 60), (300001, 1, 1), (261, 243, 1),
          (205, 131, 9)]


@pytest.mark.parametrize("nx,ny,nz", SHAPES)
def test_state_round_trip(nx, ny, nz):
    V = vah()
    n = nx * ny * nz
    rng = np.random.default_rng(nx + ny + nz)
    given = {"q": rng.random((15, n)), "e": rng.random(n), "p": rng.random(n), "u": rng.random((4, n)),
             "up": rng.random((4, n))}
    g = V.Vah(nx, ny, nz, 0.1, 0.1, 0.1, 0.01, 0.16, 0.5)
    for _ in range(2):  # a second state through the same slots
        g.set_state(3, *given.values())
        got = g.state()
        for k in given:
            assert np.array_equal(got[k], given[k]), k
        given = {k: v[..., ::-1].copy() for k, v in given.items()}
    g.close()


@pytest.mark.parametrize("nx,ny,nz", [(1, 1, 1), (41, 37, 1), (300001, 1, 1), (60, 60, 40)])
def test_batch_state_matches_the_context(nx, ny, nz):
    """Level 0 of a batch event against a context given the same primitives (the
    conformal p and u at rest are exact in both)."""
    V = vah()
    n = nx * ny * nz
    ev = dict(nx=nx, ny=ny, nz=nz, dx=0.1, dy=0.1, dz=0.1, dt=0.01, t0=0.5, etabar=0.16,
              e=1.0 + np.random.default_rng(n).random(n))
    b = V.Batch(budget_bytes=V.batch_event_bytes(nx, ny, nz) + (1 << 20), max_events=1)
    slot = admit(b, ev)
    got = b.state(slot)
    assert np.array_equal(got["e"], ev["e"])
    assert np.array_equal(got["u"][0], np.ones(n)) and not got["u"][1:].any()
    assert np.array_equal(got["u"], got["up"])
    assert np.array_equal(b.state(slot, ("p", "q"))["q"], got["q"])
    assert np.allclose(got["p"], ev["e"] / 3, rtol=1e-15, atol=0)
    b.close()
