"""vah_validity's maps reach the caller by two ways, straight from the device while the
context has no pinned slots and through them from there on: any subset of the maps holds
the values of the full call, and what is not asked for stays untouched."""
import ctypes

import numpy as np
import pytest

from tests.parity import gaussian_ic, rest_frame, vah

pytestmark = pytest.mark.gpu

_dp = ctypes.POINTER(ctypes.c_double)


@pytest.mark.parametrize("dims", [(1, 1, 1), (7, 5, 3), (41, 37, 1), (201, 201, 1)])
def test_subsets_of_the_maps(dims):
    V = vah()
    n = dims[0] * dims[1] * dims[2]
    c = V.Vah(*dims, 0.1, 0.1, 0.3, 0.01, 0.2, 0.5)
    e = gaussian_ic(*dims, dz=0.3, seed=n, peak=60.0) + 1.0
    c.set_primitives(e, *rest_frame(n), pl=e / 3)
    c.step(2)
    c.synchronize()
    full = list(c.validity().values())
    assert len(full) == 5 and all(a.size == n and np.all(np.isfinite(a)) for a in full)
    for mask in (0, 1, 2, 4, 8, 16, 5, 26, 31):
        got = [np.full(n, -1.0) for _ in range(5)]
        rc = V.lib().vah_validity(c.h, *(a.ctypes.data_as(_dp) if mask >> k & 1 else None for k, a in enumerate(got)))
        assert rc == V.VAH_OK
        for k, a in enumerate(got):
            assert np.array_equal(a, full[k].ravel()) if mask >> k & 1 else np.all(a == -1.0), (mask, k)
    c.close()
