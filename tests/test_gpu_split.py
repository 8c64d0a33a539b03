"""Forces on either side of the line where stencils change form (2^15 sites),
with ragged last groups, and thin constrained forces, whose links with two
staple sums have a launch of their own, against the FP64 oracle. FP64 1e-12,
FP32 2e-5 of the largest component (as in the parity tests)."""
import numpy as np
import pytest

import mag_amd as M
from mag_amd import ALG8, F32, F64, LINK12, LINK18

pytestmark = pytest.mark.gpu

SHAPES = [(4, 4, 4, 4), (9, 7, 11, 13), (16, 16, 16, 8), (16, 16, 16, 9), (8, 8, 4, 24)]


def check(ctx, orc, L, act, seed):
    U = orc.haar_links(L, seed)
    a = M._lib.Action(act.type, act.beta, act.c1, act.mag, act.n_stout, act.rho)
    for prec, kind, tol in ((F64, LINK18, 1e-12), (F64, LINK12, 1e-12), (F32, LINK12, 2e-5)):
        f = M.Field(ctx, L, kind, prec).upload(U)
        ref = orc.get_force(L, f.download() if prec == F32 else U, act)
        F = M.Field(ctx, L, ALG8, prec)
        M.get_force(F, f, a)
        err, big = np.abs(F.download() - ref).max(), np.abs(ref).max()
        print(f"{L} type {act.type} mag {act.mag} n {act.n_stout} prec {prec} kind {kind}: {err:.2e} of {big:.2e}",
              flush=True)
        assert err <= tol * big  # mag = 1: every link is the last of its block, all forces are zero


@pytest.mark.parametrize("L", SHAPES)
@pytest.mark.parametrize("kind,n_stout", [(0, 0), (1, 0), (0, 1), (1, 2)])
def test_force_forms(ctx, orc, L, kind, n_stout):
    check(ctx, orc, L, orc.action(kind, 6.0 if kind == 0 else 2.6, -0.331 if kind else 0.0, n_stout=n_stout), 31)


@pytest.mark.parametrize("L,mag", [((4, 4, 4, 4), 2), ((6, 6, 6, 12), 3), ((8, 4, 8, 12), 4), ((12, 12, 12, 12), 2),
                                   ((4, 4, 4, 4), 1), ((16, 16, 16, 12), 2)])
@pytest.mark.parametrize("kind", [0, 1])
def test_thin_constrained_force(ctx, orc, L, mag, kind):
    check(ctx, orc, L, orc.action(kind, 6.0 if kind == 0 else 2.6, -0.331 if kind else 0.0, mag=mag), 32)
