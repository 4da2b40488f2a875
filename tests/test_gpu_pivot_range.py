"""Pivots at the ends of the exponent range.  The reciprocal of a pivot above 2^126 (FP32;
FP64: 2^1022) is denormal: the elimination must not depend on it.

Top: every pivot of the system lies in [1, 2), so 2^126 (2^1022) times it is in the last two
binades.  Scaling by a power of four commutes with every rounding of the factorisation and the
sweeps, 1/sqrt included, so with FP32 factors two systems so scaled, both of whose tiles are
eliminated in the way for such pivots, have the same bits.  Against the unscaled system the
bounds are the repository's own: FP64 1e-12, FP32 10 sqrt(eps) relative; two mixed solutions,
each with a backward error of 1e-12 at a condition number below 20, are 8e-11 apart at most.
Both ends in a tile: a diagonal system, whose solution each operation rounds once."""
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
    f64 = mode == "plain" and T == torch.float64
    s, t = (A.dtype.type(2.0) ** e for e in ((1022, 1004) if f64 else (126, 104)))
    x, rc, info = run(A, B, d, T, mode, combined)
    assert rc == 0 and info == 0
    xs, rc, info = run(A * s, B * s, d * s, T, mode, combined)
    assert rc == 0 and info == 0
    xt, rc, info = run(A * t, B * t, d * t, T, mode, combined)
    assert rc == 0 and info == 0
    if not f64:  # (FP64's hardware estimate of 1/sqrt need not scale)
        assert np.array_equal(xs, xt)
    tol = 8e-11 if mode == "mixed" else 1e-12 if f64 else 10 * np.sqrt(np.finfo(np.float32).eps)
    assert np.abs(xs - x).max() <= tol * np.abs(x).max()


@pytest.mark.parametrize("T", [torch.float64, torch.float32])
@pytest.mark.parametrize("n", [16, 48, 64, 96, 128])
def test_both_ends(n, T):
    N, dt = 9, np.float64 if T == torch.float64 else np.float32
    top, low = (1022, -1000) if T == torch.float64 else (126, -110)
    r = np.random.default_rng(n)
    a = (r.uniform(1, 1.9, (n, N)) * 2.0 ** r.choice([top, low, 0], (n, N))).astype(dt)
    A = np.zeros((n, n, N), dtype=dt, order="F")
    A[np.arange(n), np.arange(n)] = a
    u = r.uniform(0.5, 1, (n, 1, N)).astype(dt)
    x, rc, info = run(A, np.zeros((n, n, N - 1), dtype=dt, order="F"), a[:, None] * u, T)
    assert rc == 0 and info == 0
    # 1/sqrt twice, to 1 ulp each, and three products
    assert (np.abs(x - u) <= 8 * np.finfo(dt).eps * u).all()
