"""Left singular vectors of a split at the edges of the row ranges of the
kernels that apply the reflectors (128, 256, 512 and 1024 rows), for one, an odd
and an even number of reflectors and full column rank, against LAPACK."""

import numpy as np
import pytest

from oqupy_amd.backends import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [2, 63, 64, 65, 127, 128, 129, 192, 256, 257, 511, 512, 513,
                               1023, 1024, 1025])
@pytest.mark.parametrize("r", [1, 2, 41, 130])
def test_left_vectors(m, r):
    n = r + 3
    r = min(m, r)
    rng = np.random.default_rng([m, r])
    a = rng.normal(size=(m, r)) + 1j * rng.normal(size=(m, r))
    b = rng.normal(size=(r, n)) + 1j * rng.normal(size=(r, n))
    mat = a @ b                       # rank r
    print(f"[gpu-case] left vectors {m} x {n} rank {r}", flush=True)
    u, s, svh, _ = engine.split_svd(mat, 1e-9)
    full = np.linalg.svd(mat, compute_uv=False)
    # 1e-12 as in the other SVD tests; rank r is far above the cut of 1e-9
    assert len(s) == r
    assert np.abs(s - full[:r]).max() <= 1e-12 * full[0]
    assert np.abs(u.conj().T @ u - np.eye(r)).max() <= 1e-12
    assert np.linalg.norm(u @ svh - mat) <= 1e-12 * full[0]
