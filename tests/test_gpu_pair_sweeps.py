"""The block Jacobi SVD (ranks above 126) against LAPACK: first rank, full and
ragged column blocks, an odd number of blocks, a deficient and a clustered
spectrum, values whose squares are near the ends of the range, and a matrix too
large for the tiles in LDS."""

import numpy as np
import pytest

from oqupy_amd.backends import engine

pytestmark = pytest.mark.gpu

EPSREL = 1e-9


def _unitary(rng, m, r):
    a = rng.normal(size=(m, r)) + 1j * rng.normal(size=(m, r))
    return np.linalg.qr(a)[0]


@pytest.mark.parametrize("m,n,kind,scale", [
    (127, 127, "graded", 1.0), (128, 400, "graded", 1.0), (400, 129, "graded", 1.0),
    (161, 160, "graded", 1.0), (260, 177, "pairs", 1.0), (177, 260, "deficient", 1.0),
    (300, 300, "equal", 1.0), (150, 150, "graded", 1e-140), (150, 150, "graded", 1e140),
    (1210, 1205, "graded", 1.0)])
def test_block_jacobi(m, n, kind, scale):
    rng = np.random.default_rng([m, n])
    r = min(m, n)
    s = 10.0 ** (-8.0 * np.arange(r) / (r - 1))
    if kind == "pairs":
        s = s[np.arange(r) // 2 * 2]
    elif kind == "deficient":
        s = np.where(np.arange(r) < r - 40, s, 0.0)
    elif kind == "equal":
        s = np.ones(r)
    mat = (_unitary(rng, m, r) * s) @ _unitary(rng, n, r).conj().T * scale
    print(f"[gpu-case] block jacobi {m} x {n} {kind} {scale:g}", flush=True)
    u, sv, svh, _ = engine.split_svd(mat, EPSREL)
    full = np.linalg.svd(mat, compute_uv=False)
    tail = np.sqrt(np.cumsum((full[::-1] / full[0]) ** 2)[::-1])
    k = int(np.count_nonzero(tail > EPSREL))
    # eps * sqrt(m n) * s0 is 2e-14 to 2.7e-13 s0 here; 1e-12 as in the other
    # SVD tests
    assert len(sv) == k
    assert np.abs(sv - full[:k]).max() <= 1e-12 * full[0]
    assert np.abs(u.conj().T @ u - np.eye(k)).max() <= 1e-12
    err = np.linalg.norm(u @ svh - mat) / full[0]
    assert err <= (tail[k] if k < len(full) else 0.0) + 1e-12
