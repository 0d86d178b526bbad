"""The radix-pass kernels, on grids without a paired kernel (the lists of the
paired kernels are read to say so): the plane pass in every launch shape, split
through HBM and autotuned, and the one-workgroup k column kernel with its
projector sums, launch shapes, batches, lock-step and block solvers. On grids
with a paired kernel the settings these tests turn have no effect."""
import math

import numpy as np
import pytest

from kernel_tables import paired_cubes, paired_lengths, paired_planes
from test_gpu_plane import _reference

pytestmark = pytest.mark.gpu

# (n0, n1, n2): no paired plane; the x axis without (18) and with (20, 24) a
# paired kernel; 48 x 40 and 54 x 27 unequal, 75 x 75 past 64 x 64 points.
GRIDS = ((18, 50, 50), (20, 48, 40), (24, 54, 27), (18, 75, 75))


def _thin(grid, ecut=2.0):
    """A thin cell whose y and z axes need (nearly) grid[1:] points."""
    from baandi_amd.hamiltonian import GammaSystem
    assert grid[1:] not in paired_planes()
    kmax = math.sqrt(2.0 * ecut)
    side = lambda n: (n - 1.2) * 2.0 * math.pi / (4.0 * kmax)
    rows = [[4.0, 0, 0], [0, side(grid[1]), 0], [0, 0, side(grid[2])]]
    s = GammaSystem(rows, [[0, 0, 0]], 4.0, ecut, betas=None, grid_override=grid)
    assert tuple(s.dims) == grid
    return s


def _case(grid, precision, m=5):
    import torch
    from baandi_amd import lib as L
    from baandi_amd.hamiltonian import DistributedRealHamiltonian
    s = _thin(grid)
    g = torch.Generator(device="cuda").manual_seed(grid[1])
    x = torch.randn(m, s.n, generator=g, device="cuda", dtype=torch.float64)
    x /= x.norm(dim=1, keepdim=True)
    v = torch.randn(int(np.prod(grid)), generator=g, device="cuda", dtype=torch.float64)
    prec = {"fp64": L.BD_FP64, "fp32hx": L.BD_FP32_HX, "mixed": L.BD_MIXED}[precision]
    op = DistributedRealHamiltonian(s, capacity=m, precision=prec)
    op.set_owned_potential(v)
    return s, op, x, v


def _pass(op, x, v, kept=True):
    """(H X, density, dV X from the kept fields)."""
    import torch
    y, rho, z = torch.full_like(x, float("nan")), torch.full_like(v, float("nan")), torch.zeros_like(x)
    op.apply_block(x, y)
    if kept:
        op.keep_fields(True)
    op.band_density_sum(x, np.linspace(2.0, 0.5, x.shape[0]), rho)
    if kept:
        op.apply_kept(x, v, z)
        op.keep_fields(False)
    torch.cuda.synchronize()
    return y, rho, z


def _check(s, x, v, outputs, precision):
    """Against torch's FFTs; bounds as in the plane pass's test (the kinetic term
    taken off): 100 eps of the result's norm."""
    import torch
    y, rho, z = outputs
    psi, ref = _reference(torch, s, x, v)
    w = torch.linspace(2.0, 0.5, x.shape[0], dtype=torch.float64, device="cuda").view(-1, 1, 1, 1)
    want = (w * psi * psi).sum(dim=0).reshape(-1) / s.volume
    local = y - torch.from_numpy(s.get("kinetic_orc")).cuda() * x
    bound = 100.0 * (2.0 ** -53 if precision == "fp64" else 2.0 ** -24)
    errors = [float((a - b).norm() / b.norm()) for a, b in ((local, ref), (rho, want), (z, ref))]
    print(f"[radix] {s.dims} {precision}: H·X {errors[0]:.1e} density {errors[1]:.1e} kept {errors[2]:.1e}", flush=True)
    assert max(errors) < bound


@pytest.mark.parametrize("precision", ["fp64", "fp32hx", "mixed"])
@pytest.mark.parametrize("grid", GRIDS)
def test_plane_shapes(grid, precision):
    """Every shape (256 and 512 threads, rows a chunk) gives the same bits."""
    import torch
    from baandi_amd import lib as L
    s, op, x, v = _case(grid, precision)
    assert op.plane_split() == 0
    first = _pass(op, x, v)
    _check(s, x, v, first, precision)
    taken = set()
    for threads in (256, 512):
        for chunk in (1, 4, 16, 25, grid[1]):
            try:
                op.set_plane_shape(threads, chunk)
            except L.BaandiError:
                continue  # more butterflies than the workgroup holds
            taken.add(threads)
            assert all(torch.equal(a, b) for a, b in zip(_pass(op, x, v), first)), (threads, chunk)
    assert taken == {256, 512}
    shape = op.autotune(5, reps=2)
    assert op.plane_shape() == (int(shape[0]), int(shape[1]))
    assert all(torch.equal(a, b) for a, b in zip(_pass(op, x, v), first))


@pytest.mark.parametrize("precision", ["fp64", "fp32hx", "mixed"])
@pytest.mark.parametrize("grid", GRIDS)
def test_split_plane_pass(grid, precision):
    """Planes through HBM, 1, 3 and all z lines at a time: the bits of the
    one-workgroup pass (H·X and density; the split pass keeps no fields)."""
    import torch
    s, op, x, v = _case(grid, precision)
    whole = _pass(op, x, v)
    _check(s, x, v, whole, precision)
    lines = op.plan_info()["z_planes"]
    for zb in (1, 3, min(lines, 8), 0):
        op.set_plane_split(zb)
        assert op.plane_split() == zb
        y, rho, _ = _pass(op, x, v, kept=False)
        assert torch.equal(y, whole[0]) and torch.equal(rho, whole[1]), zb


def _al(grid, betas=True, capacity=8, count=3):
    """k points of the Al cell on a grid whose columns the radix-pass kernel
    takes: not a cube, or a cube without a paired kernel."""
    from baandi_amd import workloads as W
    from baandi_amd.hamiltonian import GammaSystem
    from baandi_amd.kpoint import KPointHamiltonian
    assert len(set(grid)) > 1 or grid[0] not in paired_cubes()
    wl = W.al4()
    system = GammaSystem(wl["rows"], wl["atoms"], wl["z"], 5.0, betas=wl["betas"] if betas else (),
                         dij_ry=wl["dij_ry"] if betas else (), grid_override=grid)
    assert tuple(system.dims) == grid
    rng = np.random.default_rng(1)
    pot = 0.3 * rng.standard_normal(grid) - 0.4
    ops = [KPointHamiltonian(system, k, capacity=capacity)
           for k in ((0.0, 0.0, 0.0), (0.21, 0.13, -0.34), (0.5, 0.25, 0.0))[:count]]
    for op in ops:
        op.set_owned_potential(pot.reshape(-1))
        assert op.fused_shape()[0] > 0
    return system, ops, pot


AL_GRIDS = ((18, 18, 18), (18, 20, 24))


def _blocks(ops, m, seed):
    import torch
    rng = np.random.default_rng(seed)
    return [torch.from_numpy(rng.standard_normal((m, op.global_len()))).cuda() for op in ops]


@pytest.mark.parametrize("betas", [False, True])
@pytest.mark.parametrize("grid", AL_GRIDS)
def test_k_column_kernel_shapes(grid, betas):
    """Launch shapes and the autotuned one: the same bits; the staged passes:
    the same bits without projectors, sums in another order with them (1e-14
    of the largest value)."""
    import torch
    from baandi_amd import lib as L
    _, ops, _ = _al(grid, betas)
    for op in ops:
        x = _blocks([op], 7, 3)[0]
        y, z = torch.empty_like(x), torch.empty_like(x)
        op.apply_block(x, y)
        default = op.fused_shape()
        tried = 0
        for shape in ((256, 8, 5, 1), (256, 16, 18, 2), (512, 32, 9, 1), (512, 64, 18, 3), (1024, 64, 18, 2)):
            try:
                op.set_fused_shape(shape)
            except L.BaandiError:
                continue
            tried += 1
            op.apply_block(x, z)
            torch.cuda.synchronize()
            assert torch.equal(y, z), shape
        assert tried >= 3
        op.set_fused_shape(default)
        op.autotune(7, reps=2)
        op.apply_block(x, z)
        torch.cuda.synchronize()
        assert torch.equal(y, z)
        op.set_fused_shape((0, 0, 0, 0))
        op.apply_block(x, z)
        torch.cuda.synchronize()
        d = float((y - z).abs().max() / z.abs().max())
        print(f"[radix k] {grid} betas={betas} nk={op.nk}: {tried} shapes, staged {d:.1e}", flush=True)
        assert d < 1e-14 if betas else torch.equal(y, z)


@pytest.mark.parametrize("grid", AL_GRIDS)
def test_k_batch(grid):
    """Three spheres with projectors in one launch: the bits of each alone."""
    import torch
    from baandi_amd.kpoint import KPointBatch
    _, ops, _ = _al(grid)
    xs = [_blocks([op], m, 9)[0] for op, m in zip(ops, (5, 1, 8))]
    ys = [torch.empty_like(x) for x in xs]
    KPointBatch(ops).apply(xs, ys)
    torch.cuda.synchronize()
    for op, x, y in zip(ops, xs, ys):
        alone = torch.empty_like(x)
        op.apply_block(x, alone)
        torch.cuda.synchronize()
        assert torch.equal(y, alone)


@pytest.mark.parametrize("grid", AL_GRIDS)
def test_k_lockstep_davidson(grid):
    """The lock-step Davidson on the column kernel: each k point's own solve."""
    import torch
    from baandi_amd import lib as L, ref_davidson
    from baandi_amd.kpoint import KDavidson, as_complex, solve
    from test_gpu_kpoint import _al_starts
    bands = 8
    _, ops, _ = _al(grid, capacity=bands)
    starts = _al_starts(ops, bands, 17)
    diags = [torch.from_numpy(op.get("diagonal_static") - 0.4).cuda() for op in ops]
    o = ref_davidson.Options(bands=bands, threshold=1e-11, occupied=bands, max_iterations=200,
                             preconditioner=L.BD_PRECOND_TPA)
    outs = [(torch.empty_like(x), None) for x in starts]
    sols = KDavidson(ops, bands).solve(starts, diags, o, outs)
    for k, op in enumerate(ops):
        ref = solve(op, as_complex(starts[k]), diags[k], o)
        assert sols[k].converged.all()
        assert np.abs(sols[k].eigenvalues - ref.eigenvalues).max() < 1e-10


def test_k_block_solver():
    """The block iteration over all k points (eager and from its graph): the
    bits of each k point's own."""
    import torch
    from baandi_amd import lib as L, ref_davidson
    from baandi_amd.kpoint import KBlocks, realified_start
    nb = 16
    _, ops, _ = _al((18, 20, 24), capacity=nb)
    rng = np.random.default_rng(3)
    starts, diags, alone = [], [], []
    for op in ops:
        z = rng.standard_normal((8, op.nk)) + 1j * rng.standard_normal((8, op.nk))
        starts.append(realified_start(torch.from_numpy(z / np.linalg.norm(z, axis=1, keepdims=True)).cuda()))
        diags.append(torch.from_numpy(op.get("diagonal_static") - 0.4).cuda())
        it = ref_davidson.BlockIteration(op, nb, L.BD_PRECOND_TPA, graph=False)
        it.set_diagonal(diags[-1])
        alone.append([it.start(starts[-1])] + [it.step() for _ in range(3)])
    for graph in (False, True):
        kb = KBlocks(ops, nb, L.BD_PRECOND_TPA)
        kb.set_diagonals(diags)
        values = [kb.start(starts)] + [kb.step(1, use_graph=graph) for _ in range(3)]
        assert all(np.array_equal(values[s][k], alone[k][s]) for k in range(len(ops)) for s in range(4)), graph


def test_lists_hold_the_measured_grids():
    """The lists are read right: the grids of the cells in workloads.py."""
    assert {(72, 72), (144, 144), (36, 36)} <= paired_planes()
    assert {72, 135, 144, 36, 15} <= paired_lengths() and 18 not in paired_lengths()
    assert 25 in paired_cubes() and 18 not in paired_cubes()
