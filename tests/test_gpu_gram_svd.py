"""The Jacobi SVD on the Gram matrix (one workgroup) against LAPACK at the
edges of its range: odd and even ranks, the 16-column tiles of the Gram
matrix, the largest rank in one workgroup (126 columns) and after the
grid's QR, the first rank beyond; repeated singular values, rank
deficiency, and values whose squares are near the ends of the range."""

import numpy as np
import pytest

from oqupy_amd.backends import engine

pytestmark = pytest.mark.gpu

EPSREL = 1e-9


def _unitary(rng, m, r):
    a = rng.normal(size=(m, r)) + 1j * rng.normal(size=(m, r))
    return np.linalg.qr(a)[0]


def _check(mat, name):
    print(f"[gpu-case] gram svd {name} {mat.shape}", flush=True)
    u, s, svh, _ = engine.split_svd(mat, EPSREL)
    full = np.linalg.svd(mat, compute_uv=False)
    tail = np.sqrt(np.cumsum((full[::-1] / full[0]) ** 2)[::-1])
    k = int(np.count_nonzero(tail > EPSREL))
    # backward stability of a Jacobi SVD of a few hundred rows: a small
    # multiple of eps * sqrt(m n) * s0; 1e-12 as in the other SVD tests
    assert len(s) == k
    assert np.abs(s - full[:k]).max() <= 1e-12 * full[0]
    assert np.abs(u.conj().T @ u - np.eye(k)).max() <= 1e-12
    err = np.linalg.norm(u @ svh - mat) / full[0]
    assert err <= (tail[k] if k < len(full) else 0.0) + 1e-12


@pytest.mark.parametrize("m,n", [
    (1, 1), (2, 2), (3, 2), (5, 3), (16, 16), (40, 17), (17, 40), (33, 33),
    (64, 64), (90, 65), (96, 95), (96, 96), (130, 97), (97, 130), (300, 125),
    (126, 126), (126, 260), (127, 127), (300, 128)])
def test_graded(m, n):
    rng = np.random.default_rng([m, n])
    r = min(m, n)
    s = 10.0 ** (-8.0 * np.arange(r) / max(r - 1, 1))
    _check((_unitary(rng, m, r) * s) @ _unitary(rng, n, r).conj().T, "graded")


@pytest.mark.parametrize("n", [7, 64, 100])
@pytest.mark.parametrize("kind", ["equal", "pairs", "deficient", "zeros"])
def test_special_spectra(n, kind):
    rng = np.random.default_rng([n, len(kind)])
    s = np.ones(n)
    if kind == "pairs":
        s = 10.0 ** (-(np.arange(n) // 2) * 8.0 / n)
    elif kind == "deficient":
        s = np.where(np.arange(n) < n // 2, 0.9 ** np.arange(n), 0.0)
    mat = (_unitary(rng, n + 5, n) * s) @ _unitary(rng, n, n).conj().T
    if kind == "zeros":
        mat[:, 1::3] = 0.0
    _check(mat, kind)


@pytest.mark.parametrize("scale", [1e-140, 1e140])
@pytest.mark.parametrize("n", [20, 110])
def test_scale_limits(n, scale):
    rng = np.random.default_rng([n, 5])
    s = 10.0 ** (-8.0 * np.arange(n) / (n - 1))
    mat = (_unitary(rng, n, n) * s) @ _unitary(rng, n, n).conj().T
    _check(mat * scale, f"scale {scale:g}")


@pytest.mark.parametrize("m,n", [
    (1, 9), (64, 1), (1280, 1), (1281, 2), (1024, 16), (640, 17), (641, 17),
    (320, 33), (321, 40), (160, 65), (161, 66), (128, 126), (160, 126),
    (257, 64), (129, 80), (31, 126), (5, 120)])
def test_register_qr_edges(m, n):
    """Rows per lane of the one-workgroup QR at the limits of its variants
    (4, 8, 12, 16 and 20) for 8 to 64 lanes a column, and just beyond."""
    rng = np.random.default_rng([m, n, 1])
    r = min(m, n)
    s = 10.0 ** (-8.0 * np.arange(r) / max(r - 1, 1))
    _check((_unitary(rng, m, r) * s) @ _unitary(rng, n, r).conj().T, "qr")
