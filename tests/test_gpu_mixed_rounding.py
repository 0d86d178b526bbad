"""The mixed tier's solves keep their rounding (GammaOp::keeps_rounding): after
eight Davidson iterations of the Si8 cell the Ritz values are those recorded
when the tier's arithmetic was fixed, before the paired passes and the products
with split sums were written. 20 bands: subspaces tridiagonalised in one
workgroup; 90 bands: by cooperating workgroups.

The bound. The BF16x3 noise of a Ritz value is ~2e-5 Ha, and any change of
rounding in the solve redraws it: with the paired passes the values moved by
1e-5 and more. The same arithmetic gives the same bits; 1e-11 leaves room for
the last bits of the host's exp and erf in the set-up."""
import json
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RECORD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "mixed_ritz_si8.json")


def ritz_values(bands):
    import torch
    from baandi_amd import lib as L, ref_davidson, workloads
    from baandi_amd.field import DensityField
    from baandi_amd.hamiltonian import DistributedRealHamiltonian
    system = workloads.build(workloads.si8())
    ionic = system.get("ionic_density_re") + 1j * system.get("ionic_density_im")
    v = DensityField(system).to_grid(torch.from_numpy(ionic).cuda()).real.contiguous().view(-1)
    kinetic = system.get("kinetic_orc")
    x = np.random.default_rng(bands).standard_normal((bands, system.n)) / (1.0 + 0.25 * kinetic * kinetic)
    x /= np.sqrt(np.square(x).cumsum(axis=1)[:, -1:])  # (a fixed order of sums)
    op = DistributedRealHamiltonian(system, capacity=bands, precision=L.BD_MIXED)
    op.set_owned_potential(v)
    options = ref_davidson.Options(bands=bands, threshold=1e-9, occupied=bands, first_step=True, max_iterations=8)
    return ref_davidson.solve(op, torch.from_numpy(x).cuda(), torch.from_numpy(system.get("diagonal_static")).cuda(),
                              options).eigenvalues


@pytest.mark.parametrize("bands", [20, 90])
def test_mixed_solve_keeps_its_rounding(bands):
    with open(RECORD) as f:
        want = np.array([float.fromhex(h) for h in json.load(f)[str(bands)]])
    diff = np.abs(ritz_values(bands) - want).max()
    print(f"[mixed rounding] {bands} bands: largest difference {diff:.1e} Ha", flush=True)
    assert diff < 1e-11
