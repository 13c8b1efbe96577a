"""Truncated SVDs on both sides of the lines between the kernels' ranges (needs
a GPU), against LAPACK: the workgroups of the grid's QR for tall matrices, and
the Jacobi that follows it."""

import numpy as np
import pytest

from oqupy_amd.backends import engine

pytestmark = pytest.mark.gpu

EPSREL = 1e-9

# a column to a workgroup from 3000 rows on, up to as many columns as compute units
TALL = [(2999, 9), (3000, 9), (3000, 1), (3000, 256), (3000, 257), (9216, 3)]

# ranks up to 112 of Y = R^H with up to 512 rows by the Gram Jacobi, others blocked
JACOBI = [(112, 512), (113, 512), (112, 513), (400, 112), (400, 113), (3, 512), (3, 513),
          (1, 513), (126, 2000)]


def _unitary(rng, m, r):
    a = rng.normal(size=(m, r)) + 1j * rng.normal(size=(m, r))
    return np.linalg.qr(a)[0]


@pytest.mark.parametrize("m,n", TALL + JACOBI)
def test_routes(m, n):
    print(f"[gpu-case] svd route {m}x{n}", flush=True)
    rng = np.random.default_rng([m, n])
    r = min(m, n)
    spec = 10.0 ** (-8.0 * np.arange(r) / max(r - 1, 1))
    mat = (_unitary(rng, m, r) * spec) @ _unitary(rng, n, r).conj().T
    u, s, svh, _ = engine.split_svd(mat, EPSREL)
    full = np.linalg.svd(mat, compute_uv=False)
    tail = np.sqrt(np.cumsum((full[::-1] / full[0]) ** 2)[::-1])
    k = int(np.count_nonzero(tail > EPSREL))
    # backward stability of a Jacobi SVD: a small multiple of eps * sqrt(m n) * s0,
    # 3.5e-13 at 9216 x 257; 1e-12 as in the other SVD tests
    assert len(s) == k
    assert np.abs(s - full[:k]).max() <= 1e-12 * full[0]
    assert np.abs(u.conj().T @ u - np.eye(k)).max() <= 1e-12
    err = np.linalg.norm(u @ svh - mat) / full[0]
    assert err <= (tail[k] if k < len(full) else 0.0) + 1e-12
