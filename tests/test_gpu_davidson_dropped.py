"""H·X is queued behind the border's factor, and a rejected border drops the
product: its time is part of the solve's seconds_apply all the same, while
h_columns counts the columns the method applies H to (as the oracle does)."""
import numpy as np
import pytest

from test_gpu_davidson_scf import si2

pytestmark = pytest.mark.gpu


def test_dropped_products_are_timed():
    """29 bands in a space of 59 plane waves: the corrections soon lie in the
    basis and the factor rejects the border (pivot ratio below 2.2e-4)."""
    from baandi_amd import lib as L, ref_davidson
    from baandi_amd.hamiltonian import DistributedRealHamiltonian
    torch, s, o = si2(ecut=2.5)
    bands = 29
    pot = o.ionic_grid + 0.05 * np.cos(np.arange(o.ionic_grid.size)).reshape(o.dims)
    op = DistributedRealHamiltonian(s, capacity=bands)
    op.set_owned_potential(pot.reshape(-1))
    op.set_profiling(True)
    g = np.random.default_rng(8).standard_normal((bands, s.n))
    g /= np.linalg.norm(g, axis=1, keepdims=True)
    diag = torch.from_numpy(s.get("diagonal_static") + pot.mean()).cuda()
    options = ref_davidson.Options(bands=bands, threshold=1e-9, occupied=bands, max_iterations=40,
                                   preconditioner=L.BD_PRECOND_QE)
    record = ref_davidson.solve(op, torch.from_numpy(g).cuda(), diag, options).record
    stages = op.stage_totals()
    on_gpu = sum(v for k, v in stages.items() if k not in ("applies", "pairs", "columns")) * 1e-3
    print(f"[dropped] {record} stages {stages}", flush=True)
    # The method does drop products here ...
    assert record["repairs"] >= 1 and stages["columns"] > record["h_columns"]
    # ... and the stages' time lies within the solve's (they are its intervals).
    assert record["seconds_apply"] >= 0.999 * on_gpu
