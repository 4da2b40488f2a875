"""The device build of the smoother's blocks at the sizes where its column groups and slices
can go wrong: n that does and does not divide a work-group, observations fewer than, equal
to and more than a slice, one block (no coupling) and more blocks than work-groups.

Tolerance: entries of A are sums of n^2 + m^2 + 1 products of three factors, each product
and sum rounded, so the error is at most (2n + 2m + 4) eps times the same sums of absolute
values (FP32 plans round once more)."""
import numpy as np
import pytest
import torch

from blockstructuredsolvers_amd import build_smoother, initialize_batched
from blockstructuredsolvers_amd.workloads import SmootherModel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [torch.float64, torch.float32])
@pytest.mark.parametrize("N", [1, 2, 1100])
@pytest.mark.parametrize("n,m", [(16, 1), (16, 128), (32, 16), (48, 33), (64, 32), (96, 128),
                                 (128, 64)])
def test_blocks(n, m, N, T):
    rng = np.random.default_rng(1000 * n + m)
    if N > 2 and n > 64:
        N = 150
    model = SmootherModel(rng.standard_normal((n, n)), rng.standard_normal((m, n)),
                          rng.standard_normal((n, n)), rng.standard_normal((m, m)))
    data = initialize_batched(N, n, T, "cuda", tuned=False)
    build_smoother(data, model)
    A, B = data.A_tensor.double().cpu().numpy(), data.B_tensor.double().cpu().numpy()
    data.close()
    F, H, Q, R = (M.astype(np.longdouble) for M in (model.F, model.H, model.Qinv, model.Rinv))
    Ai, Bi = Q + F.T @ Q @ F + H.T @ R @ H, -Q @ F
    aF, aH, aQ, aR = map(np.abs, (F, H, Q, R))
    eps = np.finfo(np.float64).eps
    tA = (2 * n + 2 * m + 4) * eps * (aQ + aF.T @ aQ @ aF + aH.T @ aR @ aH)
    tB = (2 * n + 4) * eps * (aQ @ aF)
    if T == torch.float32:
        e32 = np.finfo(np.float32).eps
        tA, tB = tA + e32 * np.abs(Ai), tB + e32 * np.abs(Bi)
    assert (np.abs(A - Ai[:, :, None]) <= tA[:, :, None]).all()
    assert B.shape[2] == N - 1 and (np.abs(B - Bi[:, :, None]) <= tB[:, :, None]).all()
