"""Checkerboard demon with commuting classes two to a launch, against the
oracle's 128 classes in order: the smallest lattice (2 members per class),
members that fill a block once and a bit, and several blocks. Same bounds as
for the 8^4 lattice: equal counts, 1e-12 on links, 1e-11 on demon energies."""
import numpy as np
import pytest

import mag_amd as M
from mag_amd import F64, LINK18, REAL1

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [(4, 4, 4, 4), (8, 4, 12, 4), (4, 8, 8, 16)])
def test_two_classes_per_launch(ctx, orc, L):
    U0 = orc.haar_links(L, 181)
    f = M.Field(ctx, L, LINK18, F64).upload(U0)
    d = [M.Field(ctx, L, REAL1, F64).upload(np.zeros((int(np.prod(L)), 4))) for _ in range(4)]
    d, (acc, rej) = M.demon_checkerboard(f, 2, 1.5, 182, d)
    V = U0.copy()
    E, (oacc, orej) = orc.demon_checkerboard(L, V, 2, 1.5, 182)
    assert (acc, rej) == (oacc, orej)
    assert acc + rej == 2 * 2 * 4 * int(np.prod(L))
    assert np.abs(f.download() - V).max() < 1e-12
    for k in range(4):
        assert np.abs(d[k].download() - E[:, :, k]).max() < 1e-11
