"""The chain lengths the auto schedule takes where none is given (host only), against the
schedule of chains of three and a base of eight: below 1280 blocks it is that schedule; from
there on a level-0 chain per CU (256) remains, every block is in one chain or a separator,
and no plan needs more workspace, so a caller's workspace and the allocation-free entry
point's scratch hold what they held.  The level algorithm on it agrees with the oracle."""
import ctypes

import numpy as np
import pytest

from blockstructuredsolvers_amd import _lib as L, workloads
from chain_emulator import plan_levels, solve_system
from oracle import oracle


def workspace(N, n, nrhs, dtype, mode, explicit):
    p = ctypes.c_void_p()
    L.call("bss_plan_create", N, n, nrhs, 1, dtype, mode, 0, ctypes.byref(p))
    try:
        if explicit:
            L.call("bss_set_option", p, L.BSS_OPT_CHAIN_LEN, 3.0)
        v = ctypes.c_int64()
        L.call("bss_plan_get", p, L.BSS_Q_WORKSPACE_BYTES, ctypes.byref(v))
        return v.value
    finally:
        L.lib().bss_plan_destroy(p)


@pytest.mark.parametrize("N", [1, 7, 300, 1279, 1280, 1281, 1535, 2048, 3001, 4096, 8192, 20000])
@pytest.mark.parametrize("n", [16, 32, 48, 64, 96, 128])
def test_default_lens(N, n):
    _, levels = plan_levels(N, n)
    if N < 1280:
        assert levels == plan_levels(N, n, chain_len=3, base_max=8)[1]
    else:
        assert len(levels[0][1]) >= 256
    for NL, chains in levels:
        seen = np.zeros(NL, dtype=int)
        for start, length, _, _ in chains:
            seen[start:start + length] += 1
        assert seen.max() == 1
        at = [start for start, _, _, _ in chains]
        assert at == sorted(at)
    for (NL, chains), (below, _) in zip(levels, levels[1:]):
        assert below == NL - sum(c[1] for c in chains)
    assert len(levels[-1][1]) == 1
    for nrhs in (1, 16):
        for dtype, mode in ((L.BSS_F64, L.BSS_MODE_PLAIN), (L.BSS_F32, L.BSS_MODE_PLAIN),
                            (L.BSS_F64, L.BSS_MODE_MIXED)):
            assert workspace(N, n, nrhs, dtype, mode, False) <= \
                workspace(N, n, nrhs, dtype, mode, True)


@pytest.mark.parametrize("N,n", [(1300, 16), (1400, 64)])
def test_default_lens_match_oracle(N, n):
    s = workloads.spd_system(N, n, nrhs=2, seed=N)
    xo, info = oracle.solve_system(s.A, s.B, s.d)
    assert info == 0
    x = solve_system(s.A, s.B, s.d)
    assert np.abs(x - xo).max() <= 1e-12 * np.abs(xo).max()
    assert oracle.backward_error(s.A, s.B, x, s.d).max() <= 1e-14
