"""The one-workgroup QR at the limits of its variants (needs a GPU), against the
spectra of the matrices: 4, 8, 16, 24, 32 and 38 rows a lane with 64, 32, 16, 8
and 4 lanes a column, the last row that fits each and the first that does not;
spectra down to 1e-15 of the largest value, cut at 1e-12 and 1e-13."""

import numpy as np
import pytest

from oqupy_amd.backends import engine

pytestmark = pytest.mark.gpu


def _unitary(rng, m, r):
    a = rng.normal(size=(m, r)) + 1j * rng.normal(size=(m, r))
    return np.linalg.qr(a)[0]


def _tails(spec):
    return np.sqrt(np.cumsum(spec[::-1] ** 2)[::-1]) / spec[0]


@pytest.mark.parametrize("lanes,n", [(64, 8), (32, 16), (16, 32), (8, 64), (4, 126)])
@pytest.mark.parametrize("rows", [4, 8, 16, 24, 32, 38])
@pytest.mark.parametrize("more", [0, 1])
def test_variant_limits(lanes, n, rows, more):
    m = lanes * rows + more
    print(f"[gpu-case] qr variant {m}x{n}", flush=True)
    rng = np.random.default_rng([m, n])
    epsrel = 1e-12 if more else 1e-13
    r = min(m, n)
    decades = 15.0
    for _ in range(100):
        spec = 10.0 ** (-decades * np.arange(r) / (r - 1))
        # no tail within 5% of the cut: the values are right to about 1e-15
        if np.all(np.abs(_tails(spec) / epsrel - 1.0) > 0.05):
            break
        decades -= 0.01
    mat = (_unitary(rng, m, r) * spec) @ _unitary(rng, n, r).conj().T
    u, s, svh, _ = engine.split_svd(mat, epsrel)
    k = int(np.count_nonzero(_tails(spec) > epsrel))
    # backward stability of a Jacobi SVD of a few hundred rows: a small multiple
    # of eps * sqrt(m n) * s0; 1e-12 as in the other SVD tests, and of the values,
    # whose rounding has to stay below 5% of the cut, 5e-15
    assert len(s) == k
    assert np.abs(s - spec[:k]).max() <= 5e-15
    assert np.abs(u.conj().T @ u - np.eye(k)).max() <= 1e-12
    assert np.linalg.norm(u @ svh - mat) <= _tails(np.append(spec, 0.0))[k] + 1e-12
