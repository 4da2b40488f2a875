"""The sweeps of several right-hand sides at the widths where their product units change (up
to 4, 8 and 16 columns) and at every block size, with and without separators on either side:
against the oracle at the repository's tolerances (FP64: 1e-12 relative and backward error
1e-13; FP32: 10 sqrt(eps) relative), and the first two columns bitwise the same at every
width."""
import numpy as np
import pytest
import torch

from blockstructuredsolvers_amd import factorize, initialize_batched, solve, workloads
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [torch.float64, torch.float32])
@pytest.mark.parametrize("N,chain_len", [(1, 1), (5, 1), (23, 3)])
@pytest.mark.parametrize("n", [16, 32, 48, 64, 96, 128])
def test_widths(n, N, chain_len, T):
    dt = np.float64 if T == torch.float64 else np.float32
    s = workloads.spd_system(N, n, nrhs=16, seed=7 * n + N)
    A, B, d = (a.astype(dt).astype(np.float64, order="F") for a in (s.A, s.B, s.d))
    ref, info = oracle.solve_system(A, B, d)
    assert info == 0
    first = None
    for nrhs in (2, 4, 5, 8, 9, 16):
        data = initialize_batched(N, n, T, "cuda", nrhs=nrhs, tuned=False, chain_len=chain_len,
                                  base_max=2)
        data.A_tensor.copy_(torch.from_numpy(A.astype(dt)))
        if N > 1:
            data.B_tensor.copy_(torch.from_numpy(B.astype(dt)))
        data.d_tensor.copy_(torch.from_numpy(np.asfortranarray(d[:, :nrhs].astype(dt))))
        factorize(data)
        solve(data)
        x = data.d_tensor.cpu().numpy()
        data.close()
        first = x[:, :2].copy() if first is None else first
        assert np.array_equal(x[:, :2], first), nrhs
        rel = np.abs(x - ref[:, :nrhs]).max() / np.abs(ref[:, :nrhs]).max()
        if T == torch.float64:
            dd = np.asfortranarray(d[:, :nrhs])
            assert rel <= 1e-12 and oracle.backward_error(A, B, x, dd).max() <= 1e-13
        else:
            assert rel <= 10 * np.sqrt(np.finfo(np.float32).eps)
