"""Forces and smeared links on either side of the sizes where a stencil changes
form (8,192, 12,288, 16,384, 20,736, 24,576 and 32,768 sites, by kernel and
precision), against the FP64 oracle. FP64 1e-12, FP32 2e-5 of the largest component
(as in the parity tests)."""
import numpy as np
import pytest

import mag_amd as M
from mag_amd import ALG8, F32, F64, LINK12, LINK18

pytestmark = pytest.mark.gpu

SHAPES = [(16, 8, 8, 8), (16, 8, 8, 9), (16, 16, 8, 6), (14, 12, 10, 9), (16, 16, 8, 8), (15, 12, 10, 10),
          (12, 12, 12, 12), (14, 12, 12, 12), (16, 16, 12, 8), (16, 16, 12, 9), (16, 16, 16, 8), (18, 16, 12, 10)]


@pytest.mark.parametrize("L", SHAPES)
@pytest.mark.parametrize("kind,n_stout,mag", [(0, 0, 0), (1, 0, 0), (0, 1, 0), (1, 1, 0), (0, 0, 2)])
def test_force(ctx, orc, L, kind, n_stout, mag):
    U = orc.haar_links(L, 33)
    act = orc.action(kind, 6.0 if kind == 0 else 2.6, -0.331 if kind else 0.0, mag=mag, n_stout=n_stout)
    a = M._lib.Action(act.type, act.beta, act.c1, act.mag, act.n_stout, act.rho)
    ref = orc.get_force(L, U, act)
    for prec, fmt, tol in ((F64, LINK18, 1e-12), (F64, LINK12, 1e-12), (F32, LINK12, 2e-5)):
        f = M.Field(ctx, L, fmt, prec).upload(U)
        want = orc.get_force(L, f.download(), act) if prec == F32 else ref
        F = M.Field(ctx, L, ALG8, prec)
        M.get_force(F, f, a)
        assert np.abs(F.download() - want).max() <= tol * np.abs(want).max()


@pytest.mark.parametrize("L", SHAPES)
def test_smear(ctx, orc, L):
    U = orc.haar_links(L, 34)
    ref = orc.stout_smear(L, U, 0.1, 1)
    for prec, fmt, tol in ((F64, LINK18, 1e-12), (F64, LINK12, 1e-12), (F32, LINK12, 2e-5)):
        f = M.Field(ctx, L, fmt, prec).upload(U)
        want = orc.stout_smear(L, f.download(), 0.1, 1) if prec == F32 else ref
        out = M.Field(ctx, L, fmt, prec)
        M.stout_smear(out, f, 0.1, 1)
        assert np.abs(out.download() - want).max() <= tol
