"""Non-finite entries of a matrix handed to the split and the product are an
error wherever they are, for matrices checked on the host (up to 131071 entries)
and on the device; the same calls succeed afterwards."""

import numpy as np
import pytest

from oqupy_amd.backends import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(1, 1), (3, 5461), (129, 127), (257, 510), (256, 512), (300, 437)])
@pytest.mark.parametrize("value", [np.nan, np.inf, complex(0.0, -np.inf)])
def test_non_finite_inputs(m, n, value):
    rng = np.random.default_rng([m, n])
    mat = rng.normal(size=(m, n)) + 1j * rng.normal(size=(m, n))
    print(f"[gpu-case] input check {m} x {n} {value}", flush=True)
    for at in {(0, 0), (m - 1, n - 1), (m // 2, n // 3)}:
        bad = mat.copy()
        bad[at] = value
        with pytest.raises(engine.EngineError, match="non-finite"):
            engine.split_svd(bad, 1e-9)
        with pytest.raises(engine.EngineError, match="non-finite"):
            engine.contract(bad, mat.T.copy())
        with pytest.raises(engine.EngineError, match="non-finite"):
            engine.contract(mat.T.copy(), bad)
    # sums of n products of normal entries: eps * n * |entries| <= 1e-11
    assert np.abs(engine.contract(mat, mat.T.copy()) - mat @ mat.T).max() <= 1e-10
    u, _, svh, _ = engine.split_svd(mat, 1e-12)
    assert np.abs(u @ svh - mat).max() <= 1e-10 * np.linalg.norm(mat)
