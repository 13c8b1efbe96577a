"""The pivoted QRs compare column norms at full width (needs a GPU). The first
two pivots are two orthogonal columns whose norms differ by 2^-25, the larger
one later; every other column is orthogonal to both and smaller. Then W is the
identity and the left vector of the largest value is Q e_j, j the step at which
its column was pivoted, so its sign shows j: the reflector of step 0 gives
-sign(c[0]) c / |c|, negative in row 0, and that of step 1, after a pivot
(cos t, sin t), (-sin t, cos t), positive for t < 0."""

import numpy as np
import pytest

from oqupy_amd.backends import engine

pytestmark = pytest.mark.gpu

# one workgroup with 64 to 4 lanes a column; the grid's QR from two workgroups on
SHAPES = [(2, 2), (9, 8), (40, 16), (30, 32), (90, 64), (128, 126),
          (2600, 8), (700, 30), (200, 100), (140, 130), (1100, 200)]


@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("other", ["next", "last"])
def test_larger_norm_is_pivoted_first(m, n, other):
    print(f"[gpu-case] pivot order {m}x{n} {other}", flush=True)
    t = -0.7
    q = 1 if other == "next" else n - 1
    mat = np.zeros((m, n))
    mat[:2, 0] = 1.25 * np.cos(t), 1.25 * np.sin(t)
    mat[:2, q] = 1.25 * (1.0 + 2.0 ** -25) * np.array([-np.sin(t), np.cos(t)])
    rest = [c for c in range(1, n) if c != q][:m - 2]
    for k, c in enumerate(rest):
        mat[2 + k, c] = 0.5 * 0.98 ** k
    u, s, _, _ = engine.split_svd(mat, 1e-9)
    assert len(s) == 2 + len(rest)
    # sums of two to four terms: a few roundings of 2^-53
    assert abs(s[0] - 1.25 * (1.0 + 2.0 ** -25)) <= 1e-14
    assert abs(s[1] - 1.25) <= 1e-14
    assert abs(u[0, 0] - np.sin(t)) <= 1e-14
    assert abs(u[1, 0] + np.cos(t)) <= 1e-14
