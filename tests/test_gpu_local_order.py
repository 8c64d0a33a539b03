"""Checkerboard Metropolis against the oracle where the order of the members
changes: x3 split in slabs over the eight chiplets for every direction, for
all but direction 3, or not at all; member counts that leave the last block
partly empty. Same bounds as for the 8^4 lattice: equal counts, 1e-12 on links
(two iterations, ~50 roundings each on elements of at most 1)."""
import numpy as np
import pytest

import mag_amd as M
from mag_amd import F64, LINK18

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mag", [0, 2])
@pytest.mark.parametrize("L", [(4, 4, 4, 4), (4, 6, 4, 8), (6, 4, 10, 16), (6, 10, 4, 12), (12, 4, 6, 18)])
def test_members(ctx, orc, L, mag):
    U0 = orc.haar_links(L, 41 + mag)
    f = M.Field(ctx, L, LINK18, F64).upload(U0)
    acc, p, cp = M.local_metropolis(f, 5.7, mag, 2, 2, 0.5, 7, M.ORDER_CHECKERBOARD)
    V = U0.copy()
    oacc, op, ocp = orc.local_metropolis(L, V, 5.7, mag, 2, 2, 0.5, 7, M.ORDER_CHECKERBOARD)
    assert acc == list(oacc)
    assert sum(acc) >= 2 * 2 * 4 * int(np.prod(L))
    assert np.abs(f.download() - V).max() < 1e-12
    assert np.abs(p - op).max() < 1e-13 and np.abs(cp - ocp).max() < 1e-13
