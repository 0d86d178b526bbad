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


def solve_thin(n1, n2, precision):
    """(H X of the Ritz vectors, the vectors, their values) after two iterations
    on a thin cell (12 x points)."""
    import torch
    from baandi_amd import ref_davidson
    from baandi_amd.hamiltonian import DistributedRealHamiltonian
    from test_gpu_plane import _cell
    s = _cell(n1, n2)
    rng = np.random.default_rng(n1)
    kinetic = s.get("kinetic_orc")
    x = rng.standard_normal((4, s.n)) / (1.0 + kinetic * kinetic)
    x /= np.sqrt(np.square(x).cumsum(axis=1)[:, -1:])
    v = torch.from_numpy(rng.uniform(-0.2, 0.2, int(np.prod(s.dims)))).cuda()
    op = DistributedRealHamiltonian(s, capacity=4, precision=precision)
    op.set_owned_potential(v)
    options = ref_davidson.Options(bands=4, threshold=1e-9, occupied=4, first_step=True, max_iterations=2,
                                   return_hx=True)
    sol = ref_davidson.solve(op, torch.from_numpy(x).cuda(), torch.from_numpy(s.get("diagonal_static")).cuda(), options)
    return s, v, sol


@pytest.mark.parametrize("n1,n2", [(36, 36), (72, 72), (144, 144), (50, 50)])
def test_mixed_solve_applies_h(n1, n2):
    """H X as a mixed solve has it, on the radix passes with whole planes (36^2
    on 256 threads, 72^2 on 512), split planes (144^2), and on a plane without a
    paired kernel (50^2), against FP64. FP32 transforms (a few 2^-24 log2 N) and
    two BF16x3 products (2^-16 of a 4- or 8-term sum each): 5e-5 of the norm."""
    import torch
    from baandi_amd import lib as L
    from baandi_amd.hamiltonian import DistributedRealHamiltonian
    s, v, sol = solve_thin(n1, n2, L.BD_MIXED)
    exact = DistributedRealHamiltonian(s, capacity=4)
    exact.set_owned_potential(v)
    y = torch.empty_like(sol.eigenvectors)
    exact.apply_block(sol.eigenvectors, y)
    err = float((sol.hx - y).norm() / y.norm())
    print(f"[mixed solve] {n1}x{n2}: H X {err:.1e}", flush=True)
    assert err < 5e-5
