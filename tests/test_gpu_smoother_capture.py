"""build_smoother takes its model from host memory that is its own only until the copy is done,
so a captured copy would read other data on replay: the call is refused during capture and
works again after it."""
import numpy as np
import pytest
import torch

from blockstructuredsolvers_amd import build_smoother, initialize_batched, workloads

pytestmark = pytest.mark.gpu


def test_refused_during_capture():
    model = workloads.smoother_model(16, np.random.default_rng(3))
    data = initialize_batched(20, 16, torch.float64, "cuda", tuned=False)
    build_smoother(data, model)
    A = data.A_tensor.clone()
    with pytest.raises(RuntimeError):
        with torch.cuda.graph(torch.cuda.CUDAGraph()):
            build_smoother(data, model)
    data.A_tensor.zero_()
    build_smoother(data, model)
    assert torch.equal(data.A_tensor, A)
    data.close()
