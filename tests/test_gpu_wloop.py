"""Wilson loops where the kernel's halves and rows change form: zero and
several spatial extents, one to three permutations and six, lattices on either
side of 2^15 sites and with a ragged last block, against the oracle (1e-13)."""
import pytest

import mag_amd as M
from mag_amd import F32, F64, LINK12, LINK18

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [(4, 4, 4, 4), (5, 7, 4, 9), (16, 16, 16, 10)])
@pytest.mark.parametrize("r,T", [((1, 0, 0), 1), ((0, 0, 0), 2), ((4, 0, 0), 4), ((2, 1, 0), 3), ((1, 1, 1), 2),
                                 ((3, 2, 1), 5)])
def test_wilson_loop(ctx, orc, L, r, T):
    U = orc.haar_links(L, 61)
    for kind, prec in ((LINK18, F64), (LINK12, F64), (LINK12, F32)):
        f = M.Field(ctx, L, kind, prec).upload(U)
        ref = orc.avg_wilson_loop(L, f.download(), r, T)
        got = M.avg_wilson_loop(f, r, T)
        print(f"{L} r {r} T {T} kind {kind} prec {prec}: {got:.15e} {ref:.15e}", flush=True)
        # an average of V traces of magnitude <= 3, each rounded at 1e-16 per product
        assert abs(got - ref) < 1e-13
