"""The dynamics step kernel against the FP64 oracle at the edges of its tiles
(16 values of the future bond per workgroup, rows of the past bond in chunks
of 16 or 64) and for every Liouville dimension it is compiled for."""

import numpy as np
import pytest

import oqupy_amd as oqupy

from oracle.dynamics import compute_dynamics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3, 4])
@pytest.mark.parametrize("transforms", [False, True])
@pytest.mark.parametrize("bonds", [
    (1, 1, 15, 16, 17, 1), (1, 63, 64, 65, 1, 1), (1, 2, 130, 33, 3, 1)])
def test_dynamics_step_edges(dim, transforms, bonds):
    print(f"[gpu-case] dynamics step dim {dim} {transforms} {bonds}",
          flush=True)
    rng = np.random.default_rng([dim, len(bonds), bonds[2], int(transforms)])
    d2 = dim * dim

    def cplx(*shape):
        return rng.normal(size=shape) + 1j * rng.normal(size=shape)

    tens = [cplx(a, b, d2) / np.sqrt(2 * max(a, b))
            for a, b in zip(bonds[:-1], bonds[1:])]
    caps = [cplx(b) / np.sqrt(b) for b in bonds]
    tin = cplx(d2, d2) / dim if transforms else None
    tout = cplx(d2, d2) / dim if transforms else None
    pt = oqupy.SimpleProcessTensor(dim, dt=0.1, transform_in=tin,
                                   transform_out=tout)
    for k, ten in enumerate(tens):
        pt.set_mpo_tensor(k, ten)
    for k, cap in enumerate(caps):
        pt.set_cap_tensor(k, cap)
    ham = cplx(dim, dim)
    system = oqupy.System(ham + ham.conj().T)
    rho = cplx(dim, dim)
    dyn = oqupy.compute_dynamics(system=system, process_tensor=pt,
                                 initial_state=rho)
    props = system.get_propagators(0.1, 0.0, None, None)
    ref = np.array(compute_dynamics(props, rho, len(tens), [tens], [caps],
                                    [(tin, tout)]))
    # five steps of sums of at most 130 * 16 * 16 terms: 1e-11 relative to
    # the largest entry is far above their rounding
    assert np.abs(dyn.states - ref).max() <= 1e-11 * np.abs(ref).max()
