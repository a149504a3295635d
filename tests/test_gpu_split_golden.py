"""One step in split precision against the fields recorded before the role kernels
(tests/golden/make_split_step.py): the float terms of the sources and fluxes keep
their order and contraction, which the order of a kernel's loads decides."""
import os

import numpy as np
import pytest

from tests.golden.make_split_step import DIMS, step
from tests.parity import vah

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "split_step.npz")


@pytest.mark.parametrize("dims", DIMS)
def test_split_step_is_the_recorded_one(dims):
    """Within 1e-12 of the cell's T^tautau (e and pi smaller than it by at most 1e2, u of
    order one): the double parts may round differently by some 1e-15, while one float
    product contracted another way moves dt S / T^tautau ~ 0.02 by 6e-8 and the result
    by 1e-9."""
    want = np.load(GOLDEN)["x".join(map(str, dims))]
    got = step(vah(), dims)
    scale = np.vstack([np.broadcast_to(want[0], (16, want.shape[1])), np.ones((4, want.shape[1]))])
    err = np.abs(got - want) / scale
    assert err.max() <= 1e-12, (np.unravel_index(err.argmax(), err.shape), err.max())
