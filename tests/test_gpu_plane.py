"""The paired plane pass (plane_kernels.hpp) at every plane it is built for:
H·X, the band density and the kept-field apply on thin cells (a few x points,
y and z axes of the wanted lengths, so that the occupied lines fill half of
them as in real cells), against torch's FFTs.

Bounds. FP64: an FFT of N points errs by a few eps log2 N, and the transforms
go both ways: 100 eps of the result's norm. FP32 transforms: the same in
2^-24 relative to the local part, which is the whole result here (no
projectors, the kinetic term removed)."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EQUAL = (15, 20, 24, 25, 27, 30, 32, 36, 40, 45, 48, 54, 60, 64, 72, 80, 90, 96, 108, 120, 128, 144)
PLANES = tuple((n, n) for n in EQUAL) + tuple((u, v) for u, v in ((30, 60), (60, 30), (60, 90), (90, 60), (30, 90),
                                                                  (90, 30), (32, 64), (64, 32), (64, 96), (96, 64),
                                                                  (32, 96), (96, 32), (36, 72), (72, 36), (72, 108),
                                                                  (108, 72), (36, 108), (108, 36)))
# Lengths with no kernel of their own keep the pass-per-radix kernels.
OTHERS = ((50, 50), (40, 48))


def _cell(n1, n2, ecut=2.0):
    """Axes whose required grid lengths (4 kmax L / 2 pi and a little) are n1, n2."""
    from baandi_amd.hamiltonian import GammaSystem
    kmax = math.sqrt(2.0 * ecut)
    side = lambda n: (n - 1.2) * 2.0 * math.pi / (4.0 * kmax)
    rows = [[4.0, 0, 0], [0, side(n1), 0], [0, 0, side(n2)]]
    return GammaSystem(rows, [[0, 0, 0]], 4.0, ecut, betas=None,
                       grid_override=(12, n1, n2))


def _reference(torch, s, x, v):
    dims = tuple(s.dims)
    n = int(np.prod(dims))
    plus, minus = (torch.from_numpy(s.get(k)).cuda() for k in ("plus_index", "minus_index"))
    c = torch.complex(x[:, 1::2], x[:, 2::2]) / math.sqrt(2.0)
    g = torch.zeros(x.shape[0], n, dtype=torch.complex128, device="cuda")
    g[:, plus[1:]] = c
    g[:, minus[1:]] = c.conj()
    g[:, plus[0]] = x[:, 0].to(torch.complex128)
    psi = torch.fft.ifftn(g.view(-1, *dims), dim=(1, 2, 3), norm="forward").real

    def back(f):
        h = torch.fft.fftn(f, dim=(1, 2, 3), norm="forward").reshape(f.shape[0], -1)[:, plus]
        out = torch.empty_like(x)
        out[:, 0] = h[:, 0].real
        out[:, 1::2] = math.sqrt(2.0) * h[:, 1:].real
        out[:, 2::2] = math.sqrt(2.0) * h[:, 1:].imag
        return out

    return psi, back(psi * v.view(dims))


@pytest.mark.parametrize("precision", ["fp64", "fp32hx"])
@pytest.mark.parametrize("n1,n2", PLANES + OTHERS)
def test_plane_pass(n1, n2, precision):
    import torch
    from baandi_amd import lib as L
    from baandi_amd.hamiltonian import DistributedRealHamiltonian
    s = _cell(n1, n2)
    assert tuple(s.dims)[1:] == (n1, n2)
    m = 3  # the last pair is half empty
    g = torch.Generator(device="cuda").manual_seed(n1 * 1000 + n2)
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
    # Density and kept fields (not on the split pass, which keeps none).
    w = np.array([2.0, 0.5, 1.0])
    rho = torch.full_like(v, float("nan"))
    kept = op.plane_split() == 0
    if kept:
        op.keep_fields(True)
    op.band_density_sum(x, w, rho)
    want = (torch.from_numpy(w).cuda().view(-1, 1, 1, 1) * psi * psi).sum(dim=0).reshape(-1) / s.volume
    derr = float((rho - want).norm() / want.norm())
    kerr = 0.0
    if kept:
        z = torch.zeros_like(x)
        op.apply_kept(x, v, z)
        kerr = float((z - ref).norm() / ref.norm())
    print(f"[plane] {n1}x{n2} {precision}: H·X {err:.1e} density {derr:.1e} kept {kerr:.1e} (bound {bound:.1e})",
          flush=True)
    assert err < bound and derr < bound and kerr < bound


@pytest.mark.parametrize("n1,n2", PLANES)
def test_mixed_density(n1, n2):
    """The FP32 paired density (the mixed tier's; FP32 H·X operators keep the
    radix passes for theirs) and the kept-field apply from its fields: bounds as
    above."""
    import torch
    from baandi_amd import lib as L
    from baandi_amd.hamiltonian import DistributedRealHamiltonian
    from kernel_tables import paired_planes
    assert (n1, n2) in paired_planes()
    s = _cell(n1, n2)
    g = torch.Generator(device="cuda").manual_seed(n1 * 1000 + n2)
    x = torch.randn(3, s.n, generator=g, device="cuda", dtype=torch.float64)
    x /= x.norm(dim=1, keepdim=True)
    v = torch.randn(int(np.prod(s.dims)), generator=g, device="cuda", dtype=torch.float64)
    op = DistributedRealHamiltonian(s, capacity=3, precision=L.BD_MIXED)
    op.set_owned_potential(v)
    psi, ref = _reference(torch, s, x, v)
    kept = op.plane_split() == 0
    if kept:
        op.keep_fields(True)
    w = np.array([2.0, 0.5, 1.0])
    rho, z = torch.full_like(v, float("nan")), torch.zeros_like(x)
    op.band_density_sum(x, w, rho)
    want = (torch.from_numpy(w).cuda().view(-1, 1, 1, 1) * psi * psi).sum(dim=0).reshape(-1) / s.volume
    bound = 100.0 * 2.0 ** -24
    assert float((rho - want).norm() / want.norm()) < bound
    if kept:
        op.apply_kept(x, v, z)
        assert float((z - ref).norm() / ref.norm()) < bound
