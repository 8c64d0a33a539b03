"""Field upload and download against the host arithmetic they stand for, bit
for bit: one chunk, a ragged last block, and many chunks over all slots."""
import numpy as np
import pytest

import mag_amd as M

pytestmark = pytest.mark.gpu


def _third_row(a):
    """Rows 0 and 1 of (V, 4, 18) links completed by conj(r0 x r1), each product rounded by itself."""
    out = a.copy()
    e = [(a[..., 2 * k], a[..., 2 * k + 1]) for k in range(6)]

    def mul(x, y):
        return x[0] * y[0] - x[1] * y[1], x[0] * y[1] + x[1] * y[0]
    for j, (p, q) in enumerate([(1, 2), (2, 0), (0, 1)]):
        u, v = mul(e[p], e[3 + q]), mul(e[q], e[3 + p])
        out[..., 12 + 2 * j] = u[0] - v[0]
        out[..., 13 + 2 * j] = -(u[1] - v[1])
    return out


def _components(a):
    s2, s6 = 0.70710678118654752440, 0.40824829046386301637
    re, im = a[..., 0::2], a[..., 1::2]
    return np.stack([s2 * (re[..., 1] + re[..., 3]), s2 * (im[..., 3] - im[..., 1]), s2 * (re[..., 0] - re[..., 4]),
                     s2 * (re[..., 2] + re[..., 6]), s2 * (im[..., 6] - im[..., 2]), s2 * (re[..., 5] + re[..., 7]),
                     s2 * (im[..., 7] - im[..., 5]), s6 * (re[..., 0] + re[..., 4] - 2.0 * re[..., 8])], -1)


def _matrix(h):
    s2, s6 = 0.70710678118654752440, 0.40824829046386301637
    m = np.zeros(h.shape[:-1] + (18,))
    for (i, j), (a, b) in {(1, 3): (0, 1), (2, 6): (3, 4), (5, 7): (5, 6)}.items():
        m[..., 2 * i] = m[..., 2 * j] = s2 * h[..., a]
        m[..., 2 * i + 1], m[..., 2 * j + 1] = -s2 * h[..., b], s2 * h[..., b]
    m[..., 0] = s2 * h[..., 2] + s6 * h[..., 7]
    m[..., 8] = -s2 * h[..., 2] + s6 * h[..., 7]
    m[..., 16] = -2.0 * s6 * h[..., 7]
    return m


@pytest.mark.parametrize("dims", [(4, 4, 4, 4), (9, 7, 11, 13), (16, 16, 16, 20)])
@pytest.mark.parametrize("kind,prec", [(M.LINK18, M.F64), (M.LINK12, M.F64), (M.LINK12, M.F32), (M.ALG8, M.F64),
                                       (M.ALG8, M.F32), (M.REAL1, M.F64)])
def test_values_are_the_host_conversion(ctx, dims, kind, prec):
    v = int(np.prod(dims))
    real = np.float32 if prec == M.F32 else np.float64
    a = np.random.default_rng(5).standard_normal((v, 4) if kind == M.REAL1 else (v, 4, 18))
    f = M.Field(ctx, dims, kind, prec).upload(a)
    if kind == M.ALG8:
        want = _matrix(_components(a).astype(real).astype(np.float64))
    elif kind == M.LINK12:
        want = _third_row(a.astype(real).astype(np.float64))
    else:
        want = a
    got = f.download()
    assert np.array_equal(got, want), np.abs(got - want).max()
