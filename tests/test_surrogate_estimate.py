"""surrogate.estimate makes a network for the grids that it is given, not for its largest batch."""
import numpy as np
import pytest


@pytest.mark.parametrize("n,most", [(0, 1), (1, 1), (512, 512), (5000, 4096)])
def test_network_fits_the_grids(monkeypatch, n, most):
    from gpu_2dising_amd import surrogate as S

    made = []

    class Net:
        def __init__(self, L, max_batch):
            made.append((L, max_batch))

        def set_params(self, p):
            pass

        def predict(self, g):
            return np.zeros(len(g), np.float32)

        def close(self):
            pass

    monkeypatch.setattr(S, "Surrogate", Net)
    est, unsure, info = S.estimate(np.ones((n, 16, 16), np.int8), None)
    assert made == [(16, most)] and est.shape == (n,) and not unsure.any() and info["pred"].shape == (n,)
