"""The first calls of a network on new parameters: its Adam moments are zero when training starts,
at creation and after set_blob."""
import numpy as np
import pytest

import mlp_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hidden", [32, 128])
def test_first_training_step_on_new_parameters(hidden):
    """The first Adam step moves every parameter whose gradient is not tiny by the learning rate,
    whatever its size: m / sqrt(v) is +-1 when both moments started at zero."""
    import torch
    from hyqmom_amd.warmstart import WarmStartMLP
    rng = np.random.default_rng(6)
    X = torch.from_numpy(rng.standard_normal((500, 16)).astype(np.float32)).cuda()
    T = torch.from_numpy(rng.standard_normal((500, 2)).astype(np.float32)).cuda()
    torch.cuda.synchronize()
    lr = 2.0 ** -10
    blobs = [R.random_blob(seed, hidden=hidden) for seed in (1, 2, 3)]

    def check(m, blob):
        _, g = m.grad(X, T)
        m.train_step(X, T, lr)
        n = len(g)
        d = m.blob()[:n].astype(np.float64) - blob[:n]
        big = np.abs(g) > 1e-5  # eps 1e-8: the step is lr to 1e-3
        assert big.sum() > n // 4
        assert np.abs(d[big] + lr * np.sign(g[big])).max() < 2e-3 * lr + 2.0 ** -22

    for blob in blobs:
        m = WarmStartMLP(blob)
        check(m, blob)
        for other in blobs:  # with moments of earlier steps to clear
            m.set_blob(other)
            check(m, other)
