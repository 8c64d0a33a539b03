"""The coarse force on either side of the coarse size where its kernel changes
form (8^4 sites), with ragged last blocks and block counts rounded up over the
XCDs, against the oracle (1e-12 of the largest component)."""
import numpy as np
import pytest

import mag_amd as M
from mag_amd import ALG8, F64, LINK18
from mag_amd import multi_md as MD

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [(8, 8, 8, 8), (8, 12, 16, 10), (16, 16, 16, 16), (16, 16, 20, 16), (20, 20, 20, 20)])
def test_coarse_and_fine_force(ctx, orc, L):
    U, P = orc.haar_links(L, 71), orc.init_momentum(L, 72, 0)
    cd = MD.coarse_dims(L)
    C = orc.haar_links(cd, 73)
    mp = MD.params(0.1, 1.2)
    omp = orc.multi(0.1, 1.2)
    dU = M.Field(ctx, L, LINK18, F64).upload(U)
    dP = M.Field(ctx, L, ALG8, F64).upload(P)
    CF = M.Field(ctx, cd, ALG8, F64)
    MD.get_Cforce(CF, dU, dP, mp)
    ref = orc.multi_cforce(L, U, P, omp)
    assert np.abs(CF.download() - ref).max() <= 1e-12 * np.abs(ref).max()
    dC = M.Field(ctx, cd, LINK18, F64).upload(C)
    X = MD.xi_field(ctx, L, 1.2)
    arg = M.Arg_chmc(beta=2.6, gauge=M.Gauge(M.IWASAKI, -0.331))
    F = M.Field(ctx, L, ALG8, F64)
    MD.get_Fforce(F, dU, dC, arg, X, mp)
    xi = np.full((int(np.prod(cd)), 4), 1.2)
    ref = orc.multi_fforce(L, U, C, xi, orc.action(1, 2.6, -0.331), omp)
    assert np.abs(F.download() - ref).max() <= 1e-12 * np.abs(ref).max()
    # the sum over blocks (none of the surplus blocks may write)
    s = MD.get_xi_energy(dU, dC, X, mp)
    ref = orc.xi_energy(L, U, C, xi, omp)
    assert abs(s - ref) <= 1e-12 * (1.5 * 1.2 * 3 * 4 * np.prod(cd)) ** 0.5 * 3
