"""Pivots in the topmost binades.  The reciprocal of a pivot above 2^126 (FP32; FP64: 2^1022)
is denormal: the elimination must not depend on it.

Every pivot of the system lies in [1, 2), so 2^126 (2^1022) times it is in the last two
binades.  Scaling by a power of four commutes with every rounding of the factorisation and
the sweeps (1/sqrt included): with FP32 factors the solution has the unscaled system's bits.
(FP64's hardware estimate of 1/sqrt need not scale: the repository's 1e-12.)"""
import numpy as np
import pytest
import torch

from blockstructuredsolvers_amd import factorize, factorize_solve, initialize_batched, solve
pytestmark = pytest.mark.gpu


def system(N, n, nrhs, dtype):
    r = np.random.default_rng(91 * n + N)
    Z = r.standard_normal((n, n, N)) * (0.05 / np.sqrt(n))
    A = 1.5 * np.eye(n)[:, :, None] + Z + Z.transpose(1, 0, 2)
    B = r.standard_normal((n, n, N - 1)) * (0.1 / np.sqrt(n))
    d = r.uniform(size=(n, nrhs, N))
    return [np.asarray(a.astype(dtype), order="F") for a in (A, B, d)]


def run(A, B, d, T, mode="plain", combined=False):
    n, nrhs, N = d.shape
    data = initialize_batched(N, n, T, "cuda", nrhs=nrhs, mode=mode, tuned=False,
                              fallback=False if mode == "mixed" else None)
    for t, a in ((data.A_tensor, A), (data.B_tensor, B), (data.d_tensor, d)):
        t.copy_(torch.from_numpy(a))
    if combined:
        rc = factorize_solve(data)
    else:
        factorize(data)
        rc = solve(data)
    out = (data.d_tensor.cpu().numpy(), rc, int(np.atleast_1d(data.info())[0]))
    data.close()
    return out


@pytest.mark.parametrize("combined", [False, True])
@pytest.mark.parametrize("mode,T", [("plain", torch.float64), ("plain", torch.float32),
                                    ("mixed", torch.float64)])
@pytest.mark.parametrize("n,nrhs", [(16, 1), (32, 3), (48, 1), (64, 1), (96, 2), (128, 1)])
def test_top_of_range(n, nrhs, mode, T, combined):
    A, B, d = system(23, n, nrhs, np.float32 if T == torch.float32 else np.float64)
    s = A.dtype.type(2.0) ** (1022 if mode == "plain" and T == torch.float64 else 126)
    x, rc, info = run(A, B, d, T, mode, combined)
    assert rc == 0 and info == 0
    xs, rc, info = run(A * s, B * s, d * s, T, mode, combined)
    assert rc == 0 and info == 0
    if mode == "plain" and T == torch.float64:
        assert np.abs(xs - x).max() <= 1e-12 * np.abs(x).max()
    else:
        assert np.array_equal(xs, x)
