"""Momenta on either side of the sizes up to which the calling thread converts
them, a lattice that leaves its last run of sites ragged, and one-real-per-link
fields of the same sizes: bit for bit the host arithmetic that both ways stand for."""
import numpy as np
import pytest

import mag_amd as M
from test_gpu_transfer import _components, _matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(5, 5, 5, 5), (8, 8, 8, 8), (8, 8, 8, 9), (16, 16, 8, 8), (16, 16, 9, 8)])
@pytest.mark.parametrize("kind,prec", [(M.ALG8, M.F64), (M.ALG8, M.F32), (M.REAL1, M.F64)])
def test_values_are_the_host_conversion(ctx, dims, kind, prec):
    v = int(np.prod(dims))
    real = np.float32 if prec == M.F32 else np.float64
    a = np.random.default_rng(6).standard_normal((v, 4) if kind == M.REAL1 else (v, 4, 18))
    f = M.Field(ctx, dims, kind, prec).upload(a)
    want = a if kind == M.REAL1 else _matrix(_components(a).astype(real).astype(np.float64))
    assert np.array_equal(f.download(), want)
