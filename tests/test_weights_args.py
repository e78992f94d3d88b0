"""CPU test of the weights of a box: one for every point, whether they come as a
numpy array or as a tensor (the assignment reads N of them from memory)."""
import numpy as np
import pytest
import torch

from pyspectrum_amd import pyspectrum as P


@pytest.fixture
def on_host(monkeypatch):
    monkeypatch.setattr(P, "_device", lambda d: torch.device("cpu"))


@pytest.mark.parametrize("w", [np.ones(4), torch.ones(4), torch.ones(4, dtype=torch.float64),
                               torch.ones(0)])
def test_too_few_weights_are_refused(on_host, w):
    with pytest.raises(ValueError):
        P._weights(w, 5, 0)
    with pytest.raises(ValueError):
        P._weights_list([None, w], [3, 5], 0)


@pytest.mark.parametrize("w", [np.full(5, 2.0), torch.full((5,), 2.0), torch.full((5, 1), 2.0)])
def test_one_weight_a_point(on_host, w):
    wd, s, a = P._weights(w, 5, 0)
    assert (s, a) == (10.0, 10.0) and wd.numel() == 5
