"""The factor kernel with column strips in registers: the sizes at which its tiles, waves
and windows can go wrong -- every block size, chains of one block (no window work carried
over), of two and three (first and last block special), and longer ones (the previous
block's products in the next block's windows), with and without left and right separators.

Tolerances: the repository's own (FP64: 1e-12 relative to the oracle, backward error
1e-13; FP32: 10 sqrt(eps) relative; mixed: backward error 1e-12).  The strict lower part
of the diagonal blocks is never read by the plain path: NaN there changes no bit."""
import numpy as np
import pytest
import torch

from blockstructuredsolvers_amd import factorize, initialize_batched, solve, workloads
from oracle import oracle

pytestmark = pytest.mark.gpu


def run(A, sysm, T, mode, chain_len):
    data = initialize_batched(sysm.N, sysm.n, T, "cuda", nrhs=sysm.nrhs, mode=mode,
                              tuned=False, chain_len=chain_len, base_max=2)
    dt = np.float64 if T == torch.float64 else np.float32
    data.A_tensor.copy_(torch.from_numpy(A.astype(dt)))
    if sysm.N > 1:
        data.B_tensor.copy_(torch.from_numpy(sysm.B.astype(dt)))
    data.d_tensor.copy_(torch.from_numpy(sysm.d.astype(dt)))
    factorize(data)
    assert solve(data) == 0
    x = data.d_tensor.double().cpu().numpy()
    data.close()
    return x


@pytest.mark.parametrize("mode,T", [("plain", torch.float64), ("plain", torch.float32),
                                    ("mixed", torch.float64)])
@pytest.mark.parametrize("N,chain_len", [(1, 1), (2, 2), (3, 1), (6, 1), (8, 2), (23, 3), (41, 9)])
@pytest.mark.parametrize("n", [16, 32, 48, 64, 96, 128])
def test_strip_sizes(n, N, chain_len, mode, T):
    sysm = workloads.spd_system(N, n, nrhs=1, seed=31 * n + N)
    if T == torch.float32:
        sysm = workloads.BlockSystem(*[a.astype(np.float32).astype(np.float64, order="F")
                                       for a in (sysm.A, sysm.B, sysm.d)])
    x = run(sysm.A, sysm, T, mode, chain_len)
    ref, info = oracle.solve_system(sysm.A, sysm.B, sysm.d)
    assert info == 0
    rel = np.abs(x - ref).max() / np.abs(ref).max()
    berr = oracle.backward_error(sysm.A, sysm.B, x, sysm.d).max()
    if mode == "mixed":
        assert berr <= 1e-12
    elif T == torch.float64:
        assert rel <= 1e-12 and berr <= 1e-13
    else:
        assert rel <= 10 * np.sqrt(np.finfo(np.float32).eps)
    if mode == "plain":
        A = sysm.A.copy(order="F")
        low = np.tril_indices(n, -1)
        A[low[0], low[1], :] = np.nan
        assert np.array_equal(run(A, sysm, T, mode, chain_len), x)
