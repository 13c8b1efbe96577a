"""The one-workgroup QR's reflectors use correctly rounded square roots (needs
a GPU): a column (a, b) of a Pythagorean triple has a squared norm and a norm
without rounding, which is then the singular value to the last bit."""

import numpy as np
import pytest

from oqupy_amd.backends import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["rows", "complex"])
def test_pythagorean_columns(kind):
    print(f"[gpu-case] pythagorean {kind}", flush=True)
    for p in range(2, 12):
        for q in range(1, p):
            a, b, c = p * p - q * q, 2 * p * q, p * p + q * q
            mat = np.array([[a], [b]]) if kind == "rows" else np.array([[a + 1j * b]])
            _, s, _, _ = engine.split_svd(mat.astype(complex), 1e-9)
            assert s[0] == float(c), (a, b, c, s[0] - c)
