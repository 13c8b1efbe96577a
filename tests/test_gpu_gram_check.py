"""The passes of the Gram Jacobi (needs a GPU): a freshly formed Gram matrix
decides when the SVD is done and gives the singular values. Kahan's matrices,
on which the diagonal of the first pass's Gram matrix is off by up to 5e-11 of
the largest singular value, and passes cut short (PTE_GRAM_SWEEPS), which reach
the further passes and, of larger ranks, the hand-over to the blocked Jacobi."""

import numpy as np
import pytest

import oqupy_amd as oqupy
from oqupy_amd import operators as op
from oqupy_amd.backends import engine

from tests import models

pytestmark = pytest.mark.gpu

STATE_TOL = 1e-10


def _kahan(n, theta):
    """Kahan's matrix with column norms falling by 1e-9 a column (pivoting keeps
    the order), rows and columns with phases (the SVD is complex)."""
    s, c = np.sin(theta), np.cos(theta)
    mat = np.diag(s ** np.arange(n)) @ (np.eye(n) - c * np.triu(np.ones((n, n)), 1))
    mat = mat * (1.0 - 1e-9) ** np.arange(n)
    phase = np.exp(1j * np.arange(n) ** 2)
    return phase[:, None] * mat * phase[::-1]


def _check(mat, epsrel, name):
    print(f"[gpu-case] {name} {mat.shape}", flush=True)
    u, s, svh, _ = engine.split_svd(mat, epsrel)
    full = np.linalg.svd(mat, compute_uv=False)
    tail = np.sqrt(np.cumsum((full[::-1] / full[0]) ** 2)[::-1])
    k = int(np.count_nonzero(tail > epsrel))
    # backward stability of a Jacobi SVD of a few hundred rows: a small
    # multiple of eps * sqrt(m n) * s0; 1e-12 as in the other SVD tests
    assert len(s) == k
    assert np.abs(s - full[:k]).max() <= 1e-12 * full[0]
    assert np.abs(u.conj().T @ u - np.eye(k)).max() <= 1e-12
    err = np.linalg.norm(u @ svh - mat) / full[0]
    assert err <= (tail[k] if k < len(full) else 0.0) + 1e-12


@pytest.mark.parametrize("n,theta", [(40, 1.2), (60, 1.2), (80, 1.2), (100, 1.25),
                                     (120, 1.25)])
@pytest.mark.parametrize("rows", [0, 300])
def test_kahan(n, theta, rows):
    """In one workgroup and, with zero rows below, after the grid's QR."""
    mat = _kahan(n, theta)
    if rows:
        mat = np.concatenate([mat, np.zeros((rows + n - mat.shape[0], n))])
    _check(mat, 1e-12, f"kahan {theta}")


@pytest.mark.parametrize("m,n", [(1, 1), (9, 7), (69, 64), (105, 100), (330, 7), (330, 110)])
@pytest.mark.parametrize("sweeps", [1, 3])
@pytest.mark.parametrize("kind", ["graded", "deficient"])
def test_passes_cut_short(m, n, sweeps, kind, monkeypatch):
    rng = np.random.default_rng([m, n, sweeps])
    a = rng.normal(size=(2, m, n)) + 1j * rng.normal(size=(2, m, n))
    u, v = np.linalg.qr(a[0])[0], np.linalg.qr(a[1][:n])[0]
    s = 10.0 ** (-8.0 * np.arange(n) / max(n - 1, 1))
    if kind == "deficient":
        s[(n + 1) // 2:] = 0.0
    monkeypatch.setenv("PTE_GRAM_SWEEPS", str(sweeps))
    _check((u * s) @ v.conj().T, 1e-9, f"sweeps {sweeps} {kind}")


@pytest.mark.parametrize("sweeps", [1, 3])
def test_passes_cut_short_in_a_batch(sweeps, monkeypatch):
    """Bonds and dynamics of process tensors against the oracle, as in the other
    batch tests."""
    print(f"[gpu-case] batch, sweeps {sweeps}", flush=True)
    cases = [(0.5, 5.0, 0.2, 6, 14), (0.1, 3.0, 0.0, 4, 12), (0.7, 5.0, 0.1, 20, 26)]
    made = [models.spin_boson(a, wc, t, 0.05, k, 1e-7) for a, wc, t, k, _ in cases]
    monkeypatch.setenv("PTE_GRAM_SWEEPS", str(sweeps))
    pts = oqupy.pt_tempo_compute_batch([m[1] for m in made], 0.0,
                                       [n * 0.05 + 1e-11 for *_, n in cases],
                                       [m[2] for m in made])
    rho0 = op.spin_dm("z+")
    for (system, bath, params), pt, case in zip(made, pts, cases):
        dyn = oqupy.compute_dynamics(system=system, process_tensor=pt, initial_state=rho0)
        ref_states, ref_bonds, _ = models.oracle_pt_dynamics(system, bath, params, rho0, case[-1])
        assert list(pt.get_bond_dimensions()[1:-1]) == ref_bonds, case
        assert np.abs(dyn.states - ref_states).max() < STATE_TOL, case
