"""Davidson vector kernels at the lengths where their 16-byte pairs, 16-deep
steps and workgroup shares end, against numpy: the dot product, the subspace
matrix, the Ritz rotation, the Olsen step and the Gram-Schmidt."""
import ctypes

import numpy as np
import pytest

from capi import Device, check, lib

pytestmark = pytest.mark.gpu
EPS = np.finfo(float).eps


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 511, 513, 4097, 262_147])
@pytest.mark.parametrize("m", [1, 16, 17, 33])
def test_vector_kernels(n, m):
    print(f"[gpu] vector kernels n={n} m={m}", flush=True)
    rng = np.random.default_rng(1000 * m + n)
    ld = n + 3
    X, Y = rng.standard_normal((m, ld)), rng.standard_normal((m, ld))
    r, d = rng.standard_normal(n), 2.0 + rng.random(n)
    mo = (m + 1) // 2
    coef = rng.standard_normal((m, mo))
    with Device() as g:
        dX, dY, dr, dd, dw = g.upload(X), g.upload(Y), g.upload(r), g.upload(d), g.zeros(n)
        # sums of n products: n roundings on each side of the comparison
        out = ctypes.c_double()
        check(lib.bsg_dot(g.ctx, dr, dd, n, ctypes.byref(out)))
        assert abs(out.value - r @ d) <= 2 * n * EPS * (np.abs(r) @ d)
        G = np.zeros((m, m))
        check(lib.bsg_gram(g.ctx, dX, dY, m, n, ld, G.ctypes.data))
        x, y = X[:, :n], Y[:, :n]
        assert np.all(np.abs(G - x @ y.T) <= 2 * n * EPS * (np.abs(x) @ np.abs(y).T))
        dZ = g.upload(np.full((mo, ld), 7.0))
        check(lib.bsg_lincomb(g.ctx, dX, m, n, ld, coef.ctypes.data, mo, dZ, ld))
        Z = g.download(dZ, (mo, ld))
        assert np.all(np.abs(Z[:, :n] - coef.T @ x) <= 2 * m * EPS * (np.abs(coef).T @ np.abs(x)))
        assert np.all(Z[:, n:] == 7.0)  # nothing past a vector's end
        # Olsen: elementwise steps and one ratio of two sums of products of one
        # sign each (c > 0, e < d), so the ratio keeps n roundings
        c = np.abs(r) + 0.5
        dc, dx = g.upload(c), g.upload(np.abs(x[0]))
        check(lib.bsg_olsen_precondition(g.ctx, dx, dc, dd, 1.0, 0.0, dw, n))
        t = c / (1.0 - d)
        ratio = (t @ np.abs(x[0])) / (c @ t)
        want = (np.abs(x[0]) - ratio * c) / (1.0 - d)
        bound = (np.abs(x[0]) + abs(ratio) * c) / (d - 1.0)
        assert np.all(np.abs(g.download(dx, n) - want) <= 4 * (n + 4) * EPS * bound)
        # Gram-Schmidt against orthonormal vectors (as many as fit): the result
        # is r's remainder, normalised; its error grows with what is cancelled
        k = min(m, n - 1) if n > 1 else 0
        if k:
            q = np.linalg.qr(rng.standard_normal((n, k)))[0].T.copy()
            dq, dr2 = g.upload(q), g.upload(r)
            check(lib.bsg_gs_orthonormalise(g.ctx, dr2, dq, k, n, n, 1))
            want = r - q.T @ (q @ r)
            left = np.linalg.norm(want) / np.linalg.norm(r)
            got = g.download(dr2, n)
            assert abs(np.linalg.norm(got) - 1.0) <= 4 * n * EPS
            assert np.linalg.norm(got - want / np.linalg.norm(want)) <= 8 * (n + k) * EPS / left
