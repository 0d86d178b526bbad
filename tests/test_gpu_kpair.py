"""The paired one-workgroup-per-column k kernel (kpair.hip) at every cube it is
built for, one without it (18^3: the radix-pass kernel) and one where no column
fits a workgroup in FP64 (45^3: staged): H_k X against torch's FFTs, against the
staged passes bit for bit, and two k points of different spheres in one launch
against each alone."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

K = ((0.0, 0.0, 0.0), (0.21, 0.13, -0.34))


def _system(n, betas, ecut=2.0):
    from baandi_amd.hamiltonian import GammaSystem
    side = (n - 1.2) * 2.0 * math.pi / (4.0 * math.sqrt(2.0 * ecut))
    kw = {} if betas else dict(betas=None)
    return GammaSystem([[side, 0, 0], [0, side, 0], [0, 0, side]], [[0.1, 0.2, 0.05]], 4.0, ecut,
                       grid_override=(n, n, n), **kw)


def _reference(torch, op, dims, x, v):
    """V psi in real space and the kinetic term of interleaved columns."""
    n = int(np.prod(dims))
    index = torch.from_numpy(op.get("fft_index")).cuda()
    g = torch.zeros(x.shape[0], n, dtype=torch.complex128, device="cuda")
    g[:, index] = torch.view_as_complex(x.view(x.shape[0], -1, 2))
    psi = torch.fft.ifftn(g.view(-1, *dims), dim=(1, 2, 3), norm="forward") * v.view(dims)
    h = torch.fft.fftn(psi, dim=(1, 2, 3), norm="forward").reshape(x.shape[0], -1)[:, index]
    return torch.view_as_real(h).reshape(x.shape) + torch.from_numpy(op.get("kinetic")).cuda() * x


@pytest.mark.parametrize("precision", ["fp64", "fp32hx"])
@pytest.mark.parametrize("n", [15, 18, 20, 24, 25, 27, 30, 32, 36, 40, 45])
def test_k_column_kernel(n, precision):
    import torch
    from baandi_amd import lib as L
    from baandi_amd.kpoint import KPointBatch, KPointHamiltonian
    s = _system(n, betas=False)
    assert tuple(s.dims) == (n, n, n)
    prec = L.BD_FP64 if precision == "fp64" else L.BD_FP32_HX
    gen = torch.Generator(device="cuda").manual_seed(n)
    v = torch.randn(n ** 3, generator=gen, device="cuda", dtype=torch.float64)
    ops, xs, alone = [], [], []
    for k, m in zip(K, (5, 3)):
        op = KPointHamiltonian(s, k, capacity=m, precision=prec)
        op.set_owned_potential(v)
        x = torch.randn(m, 2 * op.nk, generator=gen, device="cuda", dtype=torch.float64)
        y = torch.full_like(x, float("nan"))
        op.apply_block(x, y)
        ref = _reference(torch, op, tuple(s.dims), x, v)
        # An FFT of N points errs by a few eps log2 N, both ways; kinetic
        # energies (of the size of V here) add theirs once.
        bound = 100.0 * (2.0 ** -53 if precision == "fp64" else 2.0 ** -24)
        err = float((y - ref).norm() / ref.norm())
        shape = op.fused_shape()
        if shape[0]:
            staged = torch.full_like(x, float("nan"))
            op.set_fused_shape((0, 0, 0, 0))
            op.apply_block(x, staged)
            op.set_fused_shape(shape)
            assert torch.equal(y, staged), (n, k)
        print(f"[k column] {n}^3 {precision} k={k} nk={op.nk} fused={shape[0] > 0}: {err:.1e} (bound {bound:.1e})",
              flush=True)
        assert err < bound
        ops.append(op)
        xs.append(x)
        alone.append(y)
    if all(op.fused_shape()[0] for op in ops):
        ys = [torch.full_like(x, float("nan")) for x in xs]
        KPointBatch(ops).apply(xs, ys)
        torch.cuda.synchronize()
        assert all(torch.equal(y, a) for y, a in zip(ys, alone))


@pytest.mark.parametrize("n", [20, 25])
def test_k_column_kernel_nonlocal(n):
    """With projectors: the staged passes add P D P^T X by GEMMs, in another
    order; sums of nk products in both (1e-14 of the largest value, as the
    radix-pass kernel's test)."""
    import torch
    from baandi_amd.kpoint import KPointHamiltonian
    s = _system(n, betas=True)
    op = KPointHamiltonian(s, K[1], capacity=4)
    op.set_owned_potential(torch.zeros(n ** 3, dtype=torch.float64, device="cuda"))
    x = torch.randn(4, 2 * op.nk, generator=torch.Generator(device="cuda").manual_seed(3), device="cuda",
                    dtype=torch.float64)
    shape = op.fused_shape()
    assert shape[0] > 0
    y, z = torch.empty_like(x), torch.empty_like(x)
    op.apply_block(x, y)
    op.set_fused_shape((0, 0, 0, 0))
    op.apply_block(x, z)
    assert float((y - z).abs().max() / z.abs().max()) < 1e-14
