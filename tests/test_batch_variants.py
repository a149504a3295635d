"""The batch engine's kernel variants (vah_batch_variant_info, vah_batch_set_variant):
the indices that callers may have stored."""
import numpy as np
import pytest

from tests.parity import vah
from tests.test_gpu_batch import admit, events_mixed, same

ACCEPTED = 6  # indices 0 to 5 have been accepted since the first variants


def test_stored_indices_still_name_a_variant():
    """Six variants; 0 and 1 are the tile and chunk they always were, 2 and 3 have seven
    rows as 32 x 7 had, odd ones below 4 march six planes."""
    vs = vah().batch_variants()
    assert len(vs) == ACCEPTED and len(set(vs)) == ACCEPTED
    assert [(v[0], v[1], v[3]) for v in vs[:2]] == [(16, 15, 3), (16, 15, 6)]
    assert [(v[1], v[3]) for v in vs[2:4]] == [(7, 3), (7, 6)]


@pytest.mark.gpu
def test_every_stored_index_is_accepted():
    V = vah()
    ev = events_mixed()[0]
    kw = dict(budget_bytes=1 << 28, max_events=2, freezeout_T_GeV=0.0)
    B = V.Batch(**kw)
    tile = V.batch_variants()[B.variant]
    assert (tile[0], tile[1], tile[3]) == (8, 7, 3)  # the default
    admit(B, ev)
    for v in range(ACCEPTED):
        B.variant = v
        assert B.variant == v
        B.step(2)
        C = V.Batch(variant=v, **kw)
        assert C.variant == v
        C.close()
    for v in (-1, ACCEPTED):
        with pytest.raises(V.VahError) as exc:
            B.variant = v
        assert exc.value.code == V.VAH_ERR_ARG
    with pytest.raises(V.VahError):
        V.Batch(variant=ACCEPTED, **kw)
    assert B.poll()[0]["nstep"] == 2 * ACCEPTED
    B.close()


@pytest.mark.gpu
def test_default_follows_the_load():
    """Without an index, few live cells run in 8 x 7 tiles and four million or more in
    16 x 15 until they fall below three; the fields are those of one explicit variant
    all the way, graphs replayed before and after each change included."""
    V = vah()
    small = events_mixed()[0]
    n = 2001  # 4.004 M cells
    x = (np.arange(n) - (n - 1) / 2) * 0.1
    e = (20.0 * np.exp(-(x[None, :] ** 2 + 2 * x[:, None] ** 2) / 2000.0) + 1.0).ravel()
    large = dict(small, nx=n, ny=n, nz=1, e=e)
    kw = dict(budget_bytes=V.batch_event_bytes(n, n, 1) + (1 << 28), max_events=3, freezeout_T_GeV=0.0,
              steps_per_graph=2)
    got = []
    for variant in (-1, 4):
        B = V.Batch(variant=variant, **kw)
        shapes = []

        def steps(k):
            B.step(k)
            tx, ty, _, kz = V.batch_variants()[B.variant]
            shapes.append((tx, ty, kz))

        a = admit(B, small)
        steps(4)
        b = admit(B, large)
        steps(5)
        states = [B.state(s) for s in (a, b)]
        B.retire(b)
        steps(3)
        states.append(B.state(a))
        got.append((shapes, states))
        B.close()
    assert got[0][0] == [(8, 7, 3), (16, 15, 6), (8, 7, 3)], got[0][0]
    assert got[1][0] == [(8, 7, 3)] * 3
    for s, t in zip(got[0][1], got[1][1]):
        assert same(s, t)
