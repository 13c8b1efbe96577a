"""Rounding errors of the truncated SVD up to rank 126 (needs a GPU) against
those of a one-sided Jacobi SVD in numpy (double precision, LAPACK's pivoted QR,
the same stopping rule): the factorisation's residual, the left vectors'
orthonormality and the singular values are to be no further off, in the median
over spectra of 1 to 12 decades."""

import numpy as np
import pytest
from scipy.linalg import qr

from oqupy_amd.backends import engine

pytestmark = pytest.mark.gpu

EPS = 2.220446049250313e-16


def _pairs(r, t):
    """Round t of the round-robin of r columns."""
    last = r + (r & 1) - 1
    q = np.arange(1, (last + 1) // 2)
    i = np.concatenate([[last], (t + q) % last])
    j = np.concatenate([[t], (t - q) % last])
    a, b = np.minimum(i, j), np.maximum(i, j)
    return a[b < r], b[b < r]


def _one_sided(mat):
    q, tri, piv = qr(mat, mode="economic", pivoting=True)
    y = tri.conj().T.copy()
    n, r = y.shape
    w = np.eye(r, dtype=complex)
    tol2 = (max(n, 16) * EPS) ** 2
    abs2 = EPS ** 2 * np.linalg.norm(y) ** 2
    rotated = True
    while rotated:
        rotated = False
        for t in range(r + (r & 1) - 1):
            a, b = _pairs(r, t)
            app = (np.abs(y[:, a]) ** 2).sum(axis=0)
            aqq = (np.abs(y[:, b]) ** 2).sum(axis=0)
            g = (y[:, a].conj() * y[:, b]).sum(axis=0)
            m2 = np.abs(g) ** 2
            need = (m2 > tol2 * app * aqq) & (m2 > abs2 * np.maximum(app, aqq))
            if not need.any():
                continue
            rotated = True
            a, b, g, d = a[need], b[need], g[need], (aqq - app)[need]
            h = np.sqrt(d * d + 4.0 * np.abs(g) ** 2)
            c = np.sqrt(0.5 + 0.5 * np.abs(d) / h)
            s = np.where(d < 0.0, -1.0, 1.0) * g / (h * c)
            for x in (y, w):
                xa, xb = x[:, a].copy(), x[:, b].copy()
                x[:, a] = c * xa - s.conj() * xb
                x[:, b] = s * xa + c * xb
    sigma = np.linalg.norm(y, axis=0)
    order = np.argsort(-sigma)
    svh = np.empty((r, n), dtype=complex)
    svh[:, piv] = y[:, order].conj().T
    return (q @ w)[:, order], sigma[order], svh


def _errors(mat, u, s, svh, true):
    k = len(s)
    return (np.linalg.norm(u @ svh - mat) / true[0],
            np.linalg.norm(u.conj().T @ u - np.eye(k)),
            np.abs(s - true[:k]).max() / true[0])


@pytest.mark.parametrize("m,n", [(24, 24), (60, 64), (88, 83), (200, 83), (126, 126)])
def test_errors_against_one_sided_jacobi(m, n):
    print(f"[gpu-case] gram accuracy {m}x{n}", flush=True)
    r = min(m, n)
    ours, model = [], []
    for decades in range(1, 13, 2):
        rng = np.random.default_rng([m, n, decades])
        a = rng.normal(size=(m, r)) + 1j * rng.normal(size=(m, r))
        b = rng.normal(size=(n, r)) + 1j * rng.normal(size=(n, r))
        spec = 10.0 ** (-decades * np.arange(r) / (r - 1))
        mat = (np.linalg.qr(a)[0] * spec) @ np.linalg.qr(b)[0].conj().T
        true = np.linalg.svd(mat, compute_uv=False)
        u, s, svh, _ = engine.split_svd(mat, 1e-15)
        ours.append(_errors(mat, u, s, svh, true))
        model.append(_errors(mat, *_one_sided(mat), true))
    ours, model = np.median(ours, axis=0), np.median(model, axis=0)
    print("  ours", ours, "numpy", model)
    assert np.all(ours <= model)
