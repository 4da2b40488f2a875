"""factor_waves is accepted without effect: a plan that names it has the schedule (from the
autotuner cache where there is an entry), the solution and the checks of one that does not."""
import numpy as np
import pytest
import torch

from blockstructuredsolvers_amd import (_lib, autotune, factorize, initialize_batched,
                                        initialize_batched_group, solve, workloads)

pytestmark = pytest.mark.gpu

TUNED = {"config": {"chain_len_levels": [9] + [2] * 15, "base_max": 2, "factor_waves": 8}, "ms": 1.0}


@pytest.mark.parametrize("n", [32, 64])
def test_schedule_is_the_tuned_one(monkeypatch, n):
    N = 200
    monkeypatch.setattr(autotune, "load_cache",
                        lambda path=None: {autotune.key(N, n, torch.float64, "plain"): TUNED})
    sysm = workloads.spd_system(N, n, seed=5)
    seen = []
    for kw in ({}, {"factor_waves": 4}, {"factor_waves": 8}):
        data = initialize_batched(N, n, torch.float64, "cuda", **kw)
        for t, a in ((data.A_tensor, sysm.A), (data.B_tensor, sysm.B), (data.d_tensor, sysm.d)):
            t.copy_(torch.from_numpy(a))
        factorize(data)
        assert solve(data) == 0
        seen.append((data.nchains, data.d_tensor.cpu().numpy()))
        data.close()
        group = initialize_batched_group([N, N], n, torch.float64, "cuda", **kw)
        seen[-1] += (group.nchains,)
        group.close()
    assert seen[0][0][0] == 20  # chains of nine
    for other in seen[1:]:
        assert other[0] == seen[0][0] and other[2] == seen[0][2]
        assert np.array_equal(other[1], seen[0][1])
    with pytest.raises(_lib.BssError):
        initialize_batched(N, n, torch.float64, "cuda", factor_waves=5)
