"""Wilson loops where one thread per loop takes them (no spatial extent; bent
loops of single-precision links on long lattices) and where x3 is walked by
eights, against the oracle (1e-13); and on lattices large enough for the other
lines of that rule, 12-real links against 18-real ones, whose loops two
wavefronts form, from the same seed."""
import pytest

import mag_amd as M
from mag_amd import F32, F64, LINK12, LINK18

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [(16, 16, 12, 11), (8, 16, 8, 36), (9, 11, 10, 37)])
@pytest.mark.parametrize("r,T", [((0, 0, 0), 1), ((0, 0, 0), 2), ((0, 0, 0), 3), ((1, 1, 1), 2), ((2, 1, 0), 2)])
def test_against_oracle(ctx, orc, L, r, T):
    U = orc.haar_links(L, 62)
    for kind, prec in ((LINK18, F64), (LINK12, F64), (LINK12, F32)):
        f = M.Field(ctx, L, kind, prec).upload(U)
        ref = orc.avg_wilson_loop(L, f.download(), r, T)
        # an average of V traces of magnitude <= 3, each rounded at 1e-16 per product
        assert abs(M.avg_wilson_loop(f, r, T) - ref) < 1e-13


@pytest.mark.parametrize("L", [(24, 24, 24, 32), (32, 32, 32, 32), (32, 32, 32, 48)])
@pytest.mark.parametrize("r,T", [((1, 0, 0), 1), ((3, 0, 0), 1), ((1, 1, 0), 1), ((1, 1, 1), 2), ((2, 2, 2), 1)])
def test_formats_agree(ctx, L, r, T):
    w = {}
    for kind, prec in ((LINK18, F64), (LINK12, F64), (LINK12, F32)):
        f = M.Field(ctx, L, kind, prec).haar(63)
        w[kind, prec] = M.avg_wilson_loop(f, r, T)
    assert abs(w[LINK12, F64] - w[LINK18, F64]) < 1e-13
    # links of 2^-24 relative rounding, at most 12 of them per loop, averaged over V loops of magnitude <= 3
    assert abs(w[LINK12, F32] - w[LINK18, F64]) < 3 * 12 * 6e-8
