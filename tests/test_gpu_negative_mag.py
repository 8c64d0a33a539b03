"""The thin force with a negative block size, on either side of 2^15 sites,
against the oracle, whose link classes take it too: every link is written.
FP64 1e-12, FP32 2e-5 of the largest component (as in the parity tests)."""
import numpy as np
import pytest

import mag_amd as M
from mag_amd import ALG8, F32, F64, LINK12, LINK18

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [(4, 4, 4, 4), (6, 6, 6, 12), (16, 16, 16, 9)])
@pytest.mark.parametrize("mag", [-2, -3])
@pytest.mark.parametrize("kind", [0, 1])
def test_every_link_is_written(ctx, orc, L, mag, kind):
    U = orc.haar_links(L, 51)
    act = orc.action(kind, 6.0 if kind == 0 else 2.6, -0.331 if kind else 0.0, mag=mag)
    a = M._lib.Action(act.type, act.beta, act.c1, act.mag, act.n_stout, act.rho)
    for prec, fmt, tol in ((F64, LINK18, 1e-12), (F32, LINK12, 2e-5)):
        f = M.Field(ctx, L, fmt, prec).upload(U)
        ref = orc.get_force(L, f.download() if prec == F32 else U, act)
        F = M.Field(ctx, L, ALG8, prec).upload(orc.init_momentum(L, 52, 0))
        M.get_force(F, f, a)
        assert np.abs(F.download() - ref).max() <= tol * np.abs(ref).max()
