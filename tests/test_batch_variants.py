"""The batch engine's kernel variants (vah_batch_variant_info, vah_batch_set_variant):
the indices that callers may have stored."""
import pytest

from tests.parity import vah
from tests.test_gpu_batch import admit, events_mixed

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
