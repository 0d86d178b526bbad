"""The paired x pass (stick.hip) at every length it is built for, and two that
keep the pass-per-radix kernels: H·X, the band density and the kept-field apply
on long cells (the x axis of the wanted length, 12 points in y and z), against
torch's FFTs, at column counts that leave a pair half empty, deal the pairs to
the XCDs whole (16 columns) or tile by tile (3 and 21)."""
import math

import numpy as np
import pytest

from test_gpu_plane import _reference

pytestmark = pytest.mark.gpu

LENGTHS = (15, 20, 24, 25, 27, 30, 32, 36, 40, 45, 48, 50, 54, 60, 64, 72, 75, 80, 81, 90, 96, 100, 108, 120, 128, 135,
           144, 150, 160)
OTHERS = (16, 18)


def _cell(n0, ecut=2.0):
    from baandi_amd.hamiltonian import GammaSystem
    kmax = math.sqrt(2.0 * ecut)
    rows = [[(n0 - 1.2) * 2.0 * math.pi / (4.0 * kmax), 0, 0], [0, 5.0, 0.0], [0, 0, 6.0]]
    return GammaSystem(rows, [[0, 0, 0]], 4.0, ecut, betas=None, grid_override=(n0, 12, 12))


@pytest.mark.parametrize("precision", ["fp64", "fp32hx"])
@pytest.mark.parametrize("n0,m", [(n, (3, 16, 21)[i % 3]) for i, n in enumerate(LENGTHS)] + [(n, 3) for n in OTHERS])
def test_stick_pass(n0, m, precision):
    """Bounds as in the plane pass's test: 100 eps of the result's norm."""
    import torch
    from baandi_amd import lib as L
    from baandi_amd.hamiltonian import DistributedRealHamiltonian
    s = _cell(n0)
    assert s.dims[0] == n0
    g = torch.Generator(device="cuda").manual_seed(n0)
    x = torch.randn(m, s.n, generator=g, device="cuda", dtype=torch.float64)
    x /= x.norm(dim=1, keepdim=True)
    v = torch.randn(int(np.prod(s.dims)), generator=g, device="cuda", dtype=torch.float64)
    op = DistributedRealHamiltonian(s, capacity=m, precision=L.BD_FP64 if precision == "fp64" else L.BD_FP32_HX)
    op.set_owned_potential(v)
    y = torch.full_like(x, float("nan"))
    op.apply_block(x, y)
    psi, ref = _reference(torch, s, x, v)
    local = y - torch.from_numpy(s.get("kinetic_orc")).cuda() * x
    bound = 100.0 * (2.0 ** -53 if precision == "fp64" else 2.0 ** -24)
    err = float((local - ref).norm() / ref.norm())
    w = np.linspace(2.0, 0.5, m)
    rho = torch.full_like(v, float("nan"))
    op.keep_fields(True)
    op.band_density_sum(x, w, rho)
    want = (torch.from_numpy(w).cuda().view(-1, 1, 1, 1) * psi * psi).sum(dim=0).reshape(-1) / s.volume
    derr = float((rho - want).norm() / want.norm())
    z = x.clone()
    op.apply_kept(x, v, z)
    kerr = float((z - x - ref).norm() / ref.norm())
    print(f"[stick] {n0} m={m} {precision}: H·X {err:.1e} density {derr:.1e} kept {kerr:.1e} (bound {bound:.1e})",
          flush=True)
    assert err < bound and derr < bound and kerr < bound
