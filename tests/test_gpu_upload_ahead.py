"""Link uploads on either side of the chunk size up to which a block's loads are
all on their way at once (1,024 sites), with ragged last blocks: bit for bit what
was sent."""
import numpy as np
import pytest

import mag_amd as M
from test_gpu_transfer import _components, _matrix, _third_row

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(8, 8, 8, 16), (9, 9, 9, 12), (9, 7, 13, 11), (12, 12, 11, 13)])
@pytest.mark.parametrize("kind,prec", [(M.LINK18, M.F64), (M.LINK12, M.F64), (M.LINK12, M.F32), (M.ALG8, M.F64)])
def test_upload(ctx, dims, kind, prec):
    a = np.random.default_rng(7).standard_normal((int(np.prod(dims)), 4, 18))
    if kind == M.ALG8:  # Hermitian traceless, so that its components carry all of it
        a = _matrix(_components(a))
        want = _matrix(_components(a))
    else:
        a = a.astype(np.float32).astype(np.float64) if prec == M.F32 else a
        want = a if kind == M.LINK18 else _third_row(a)
    assert np.array_equal(M.Field(ctx, dims, kind, prec).upload(a).download(), want)
