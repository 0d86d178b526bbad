"""The FP64 GEMM kernels at the edges of their tiles: every tile and split the
dispatch can pick, remainders in M, N and k, odd leading dimensions and
operands that start at an odd double, against NumPy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# NN: short products (16- and 32-wide), then the 64 rb x 16 nb tiles in the
# order of the dispatch, each with ragged rows, columns and k.
NN = [(1, 1, 3), (41, 13, 238), (319, 321, 37), (4719, 9, 47), (16381, 3, 98), (4678, 294, 12), (15720, 33, 48),
      (7773, 155, 37), (14853, 279, 10), (3516, 225, 41), (8499, 131, 33), (5390, 293, 30), (11946, 437, 15),
      (8623, 381, 18), (12800, 16, 1040)]
# TN: short products, then split sums over tall k.
TN = [(1, 71, 180), (347, 441, 43), (17, 16, 1024), (16, 17, 1025), (1, 155, 1683), (6, 23, 34836), (9, 352, 2582),
      (3, 194, 27544), (3, 255, 18985), (365, 105, 1983), (201, 33, 19423), (82, 104, 21395), (160, 160, 20001),
      (640, 288, 2047), (1, 1, 5000)]


@pytest.mark.parametrize("trans_a,M,N,K", [(0, *s) for s in NN] + [(1, *s) for s in TN])
def test_fp64_gemm_tiles(trans_a, M, N, K):
    """alpha A B + beta C against NumPy to 4e-16 (2 + log2 K) of sum |a||b|
    (sums in short chains, a few roundings of the largest partial sum each),
    rows between M and the leading dimension of C untouched."""
    import torch
    from baandi_amd import lib as L
    lib = L.load()
    rng = np.random.default_rng(M + 7 * N + 13 * K)
    lda, ldb, ldc = (K if trans_a else M) + 3, K + 2, M + 1
    ka, kb = (K, M) if trans_a else (M, K)
    A = rng.standard_normal((lda, kb))
    B = rng.standard_normal((ldb, N))
    C = rng.standard_normal((ldc, N))
    a = A[:ka].T if trans_a else A[:ka]
    ref = 1.25 * (a @ B[:K]) - 0.5 * C[:M]
    # One double in front: every column starts at an address of its own parity.
    up = lambda x: torch.from_numpy(np.concatenate([[np.nan], x.ravel(order="F")])).cuda()
    Ad, Bd, Cd = up(A), up(B), up(C)
    at = lambda t: t[1:].data_ptr()
    work = torch.empty(max(1, lib.bd_gemm_workspace(0, trans_a, M, N, K)), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    print(f"[gemm] trans_a={trans_a} {M}x{N}x{K}", flush=True)
    L.check(lib.bd_gemm_dev(0, trans_a, M, N, K, 1.25, at(Ad), lda, at(Bd), ldb, -0.5, at(Cd), ldc, L.ptr(work)))
    out = Cd[1:].cpu().numpy().reshape(N, ldc).T
    assert (out[M:] == C[M:]).all()
    bound = 4e-16 * (2.0 + np.log2(K)) * (1.25 * (np.abs(a) @ np.abs(B[:K])) + np.abs(C[:M]))
    assert (np.abs(out[:M] - ref) <= bound).all(), float((np.abs(out[:M] - ref) / bound).max())
