"""Served batches on either side of the number of chains where their stencils
change form (split by planes, or one thread per link), and with chains left over
from whole rounds of eight, against Chain.run: the same bits."""
import pytest

import mag_amd as M
from mag_amd import F32, F64, IWASAKI, WILSON
from mag_amd import serving as SV

pytestmark = pytest.mark.gpu

CASES = [((4, 4, 4, 4), 9), ((4, 4, 4, 4), 64), ((5, 7, 4, 9), 13), ((5, 7, 4, 9), 27), ((8, 8, 8, 8), 3),
         ((8, 8, 8, 8), 4), ((8, 8, 8, 8), 9), ((12, 12, 12, 10), 2)]


@pytest.mark.parametrize("L,n", CASES)
@pytest.mark.parametrize("prec,recon12", [(F32, True), (F64, False), (F64, True)])
@pytest.mark.parametrize("act,n_stout,mag", [(WILSON, 0, 0), (IWASAKI, 0, 0), (WILSON, 1, 0), (IWASAKI, 2, 0), (IWASAKI, 0, 2)])
def test_batch_equals_chain(ctx, L, n, prec, recon12, act, n_stout, mag):
    if mag and any(d % mag for d in L):
        pytest.skip("extents not multiples of the block size")
    beta, c1 = (6.0, 0.0) if act == WILSON else (2.6, -0.331)
    srv = SV.Server(ctx)
    ids = []
    for i in range(n):
        r = SV.request(L, act, beta, c1, n_stout, 0.1, 1, n_md=1, tau=0.05, seed=11 + i, precision=prec,
                       num_forced_accept=1, recon12=recon12, links_seed=100 + i)
        r.act.mag = mag
        ids.append(srv.submit(r))
    srv.run_until_idle()
    got = [srv.results(i)[0][0] for i in ids]
    srv.close()
    arg = M.Arg_chmc(mag=mag, trajectory_length=1, dt=0.05, beta=beta, gauge=M.Gauge(act, c1), n_stout=n_stout,
                     rho=0.1, num_forced_accept_step=1)
    for i in (0, n // 2, n - 1):
        ch = M.Chain(ctx, L, arg, seed=11 + i, precision=prec, recon12=recon12)
        ch.haar(100 + i)
        r = ch.run(1)[0]
        assert (r.h_old, r.h_new, r.avg_plaq) == (got[i].h_old, got[i].h_new, got[i].avg_plaq)
