"""Every tile shape of the batch engine in both precisions, at the edges of all its
tiles, and the autotuner, which may pick any of them: each event against the
single-lattice path, and the variants against each other bit for bit (their per-cell
code is the same template)."""
import numpy as np
import pytest

from tests.parity import gaussian_ic, vah
from tests.test_gpu_batch import admit, same, single, table, worst

pytestmark = pytest.mark.gpu

# one cell under, on and over 8, 16, 7 and 15 rows and columns, two and more tiles
DIMS = [(7, 6, 1), (8, 7, 1), (9, 8, 1), (15, 14, 1), (16, 15, 1), (17, 16, 1), (33, 22, 1), (1, 17, 1),
        (7, 8, 2), (9, 6, 7), (15, 16, 4), (16, 7, 3), (17, 15, 6), (18, 13, 13)]


def events():
    out = []
    for i, (nx, ny, nz) in enumerate(DIMS):
        e = np.maximum(gaussian_ic(nx, ny, nz, dz=0.3, seed=40 + i, peak=60.0, tilt=0.2), 1.0)
        out.append(dict(nx=nx, ny=ny, nz=nz, dx=0.1, dy=0.1, dz=0.3, dt=0.01, t0=0.5, etabar=0.16, e=e))
    return out


def check(got, ref, tau, precision, label):
    if precision == 0:
        err = worst(got, ref, tau)
        assert err <= 1e-12, (label, err)
    else:  # float terms: the split form's bound on e and u
        assert np.max(np.abs(got["e"] - ref["e"]) / ref["e"]) < 1e-4, label
        assert np.max(np.abs(got["u"] - ref["u"]) / ref["u"][0]) < 1e-4, label


@pytest.fixture(scope="module")
def reference():
    """The events' fields after so many steps: the single-lattice FP64 path (which
    test_gpu_tiles compares with the oracle at these edges)."""
    kept = {}

    def at(steps):
        if steps not in kept:
            kept[steps] = [single(ev, steps, table()) for ev in events()]
        return kept[steps]

    return at


@pytest.fixture(scope="module")
def first():
    """{precision: the events' fields of variant 0}"""
    return {}


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "split"])
@pytest.mark.parametrize("variant", range(6))
def test_variant_at_tile_edges(reference, first, variant, precision):
    V = vah()
    steps = 6
    B = V.Batch(budget_bytes=1 << 28, max_events=len(DIMS), eos_table=table(), freezeout_T_GeV=0.0, steps_per_graph=3,
                variant=variant, precision=precision)
    slots = [admit(B, ev) for ev in events()]
    B.step(steps)
    taus = {s["slot"]: s["tau"] for s in B.poll()}
    states = [B.state(s) for s in slots]
    B.close()
    for dims, s, got, ref in zip(DIMS, slots, states, reference(steps)):
        check(got, ref, taus[s], precision, (variant, dims))
    for dims, got, ref in zip(DIMS, states, first.setdefault(precision, states)):
        assert same(got, ref), (variant, dims)


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "split"])
def test_autotune_steps_are_real_steps(reference, precision):
    V = vah()
    nv = len(V.batch_variants())
    B = V.Batch(budget_bytes=1 << 28, max_events=len(DIMS), eos_table=table(), freezeout_T_GeV=0.0, steps_per_graph=3,
                precision=precision)
    slots = [admit(B, ev) for ev in events()]
    best, ms = B.autotune(1)
    assert B.variant == best and 0 <= best < nv and len(ms) == nv and np.all(np.asarray(ms) > 0)
    st = {s["slot"]: s for s in B.poll()}
    steps = 2 * nv  # one untimed and one timed step of each variant
    for dims, s, ref in zip(DIMS, slots, reference(steps)):
        assert st[s]["nstep"] == steps
        check(B.state(s), ref, st[s]["tau"], precision, dims)
    B.close()
