"""The FP64 residual pass of mixed mode, at the sizes where its lane map, chunks, wave and
item ranges can go wrong: every block size; one block, fewer blocks than a work-group has
waves, a full item, one more, several items.  One refinement step with no fallback leaves
an iterate whose backward error (about 1e-8) the pass measured; it is compared with the
same figure in extended precision.  The first solve after a factorisation also measures
||M||, the second does not.

Tolerance: each entry of the residual is a sum of 3n + 1 products and d, so its error is at
most (3n + 4) eps (||M|| ||x|| + ||d||), and the backward error, a ratio with that
denominator, is off by no more than (3n + 8) eps with its own roundings.  Diagonal blocks
are read in their upper triangle only: NaN in the strict lower part changes no bit."""
import numpy as np
import pytest
import torch

from blockstructuredsolvers_amd import factorize, initialize_batched, solve, workloads

pytestmark = pytest.mark.gpu


def measured(A, sysm):
    """[(x, device backward error)] of two one-step solves on one factorisation."""
    data = initialize_batched(sysm.N, sysm.n, torch.float64, "cuda", nrhs=sysm.nrhs,
                              mode="mixed", tuned=False, tol=1e-30, max_iters=1,
                              fallback=False)
    data.A_tensor.copy_(torch.from_numpy(A))
    if sysm.N > 1:
        data.B_tensor.copy_(torch.from_numpy(sysm.B))
    out = []
    for k in range(2):
        data.d_tensor.copy_(torch.from_numpy(sysm.d))
        if k == 0:
            factorize(data)
        solve(data)
        out.append((data.d_tensor.cpu().numpy(), data.backward_error()[0]))
    data.close()
    return out


def berr_extended(A, B, x, d):
    L = np.longdouble
    A, B, x, d = (np.moveaxis(a.astype(L), -1, 0) for a in (A, B, x, d))
    r = d - A @ x
    rows = np.abs(A).sum(axis=2)
    if len(B):
        r[:-1] -= B @ x[1:]
        r[1:] -= B.transpose(0, 2, 1) @ x[:-1]
        rows[:-1] += np.abs(B).sum(axis=2)
        rows[1:] += np.abs(B).sum(axis=1)
    den = rows.max() * np.abs(x).max(axis=(0, 1)) + np.abs(d).max(axis=(0, 1))
    return (np.abs(r).max(axis=(0, 1)) / den).astype(np.float64)


@pytest.mark.parametrize("nrhs", [1, 3, 16])
@pytest.mark.parametrize("N", [1, 2, 3, 6, 32, 33, 71])
@pytest.mark.parametrize("n", [16, 32, 48, 64, 96, 128])
def test_residual(n, N, nrhs):
    sysm = workloads.spd_system(N, n, nrhs=nrhs, seed=17 * n + N)
    A = 0.5 * (sysm.A + sysm.A.transpose(1, 0, 2))
    low = np.tril_indices(n, -1)
    An = A.copy(order="F")
    An[low[0], low[1], :] = np.nan
    got, got_nan = measured(A, sysm), measured(An, sysm)
    for (x, berr), (xn, bn) in zip(got, got_nan):
        ref = berr_extended(A, sysm.B, x, sysm.d)
        assert (ref > 1e-10).all()  # a figure well above the rounding errors
        assert np.abs(berr - ref).max() <= (3 * n + 8) * np.finfo(np.float64).eps
        assert np.array_equal(x, xn) and np.array_equal(berr, bn)
