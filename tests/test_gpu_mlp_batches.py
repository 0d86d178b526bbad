"""Loss and gradient of the learned preconditioner where the split of a batch
over workgroups and waves can go wrong: fewer groups of 16 rows than waves,
bands that end inside a wave's run of groups, rows short of a group, one band,
and more bands than the loss kernel's waves, against the oracle."""
import numpy as np
import pytest

from test_gpu_mlp import _pairs_dev, _synthetic_pairs, _theta

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,batch", [(3, 2), (16, 1), (17, 5), (259, 9), (2600, 1), (1500, 6)])
def test_gradient_splits(n, batch):
    from oracle import mlp as M
    from baandi_amd.learned import Network, loss_and_grad
    th = _theta(5)
    g, R, Tg, scal = _synthetic_pairs(n, batch + 1, n)
    net = Network(th)
    bands = list(range(batch, 0, -1))
    loss, grad = loss_and_grad(net, _pairs_dev(g, R, Tg, scal), bands)
    again = loss_and_grad(net, _pairs_dev(g, R, Tg, scal), bands)
    assert loss == again[0] and bool((grad == again[1]).all())
    ref_batch = [(g.astype(np.float64), *(float(v) for v in scal[b]), R[b].astype(np.float64),
                  Tg[b].astype(np.float64)) for b in bands]
    ref_loss, ref_grad = M.loss_and_grad(th, ref_batch, bf16=True)
    gerr = np.linalg.norm(grad.cpu().numpy() - ref_grad) / np.linalg.norm(ref_grad)
    print(f"[mlp split] n={n} batch={batch}: loss {loss:.8f} ({ref_loss:.8f}), gradient {gerr:.1e}", flush=True)
    # The oracle rounds to bf16 as the kernels do; what is left are FP32 sums
    # and bf16 values that a last-bit difference moves by 2^-8, a few in each
    # sum: the bounds of the 700-row gradient test.
    assert abs(loss - ref_loss) < 1e-5 * max(abs(ref_loss), 1e-3)
    assert gerr < 5e-3
