"""Forms by size that the tests of the plain and fast modes leave out: the learned mode's planes,
spread over waves and in turn, with network seeds; and the weight gradients' parts, 64 of 256
rows at 16384 rows, the most there are, and longer ones from one row more on (16417 rows make
58 of 288)."""
import numpy as np
import pytest

import mlp_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [0, 2])
def test_learned_step_forms_agree(shape):
    """A state without variation in z is the same in every plane of any depth (Mz = M exactly; dt is
    dtmax); 1599 cells a plane, depths on both sides of the grids from which a wave takes all
    planes of its cells (pass 1 81920 cells; pass 2 131072)."""
    import hyqmom_amd as H
    from hyqmom_amd.ensemble import jets_params
    from hyqmom_amd.warmstart import DEFAULT_MODEL, WarmStartMLP
    p0 = dict(jets_params((41, 39, 4), 1.5, 0.01, "mixed_learned"), dtmax=1e-4)
    M0 = H.initial_state(p0)[:, :, 2:3, :]
    net = WarmStartMLP.load(DEFAULT_MODEL)
    net.set_shape(shape)
    out = {}
    for Nz in (3, 51, 52, 81, 83):
        s = H.Solver(dict(p0, Nz=Nz))
        s.set_warm_start(net)
        s.set_state(np.asfortranarray(np.repeat(M0, Nz, axis=2)))
        s.run(10.0, 4)
        M = s.get_state()
        it = (s.flags() >> 16) & 0xFFF
        s.close()
        assert np.array_equal(M, np.repeat(M[:, :, :1, :], Nz, axis=2))
        out[Nz] = M[:, :, 0, :], it[:41 * 39]
    assert not np.array_equal(out[3][0], M0[:, :, 0, :])
    for Nz in out:
        assert np.array_equal(out[3][0], out[Nz][0]), Nz
        # the same seeds take the same iterations
        assert np.array_equal(out[3][1], out[Nz][1]), Nz


@pytest.mark.parametrize("hidden", [32, 128])
@pytest.mark.parametrize("n", [16384, 16385])
def test_gradient_at_the_most_parts(n, hidden):
    """As test_gradient_at_the_edges_of_its_splits: the bound of test_gradient_matches_reference,
    with the last rows' targets made to dominate, so that a part left out shows."""
    import torch
    from hyqmom_amd.warmstart import WarmStartMLP
    blob = R.random_blob(23, hidden=hidden)
    rng = np.random.default_rng(24 + n)
    X = rng.standard_normal((n, 16)).astype(np.float32)
    T = rng.standard_normal((n, 2)).astype(np.float32) * 0.5
    T[-10:] *= 1000.0
    m = WarmStartMLP(blob)
    Xd, Td = torch.from_numpy(X).cuda(), torch.from_numpy(T).cuda()
    torch.cuda.synchronize()
    loss, g = m.grad(Xd, Td)
    lref, gref = R.loss_and_grad(blob, X, T, use_bf16=True)
    assert abs(loss - lref) <= 1e-3 * lref, (loss, lref)
    o = 0
    for name, shp in R.shapes(hidden):
        k = int(np.prod(shp))
        a, b = g[o:o + k], gref[o:o + k]
        o += k
        nb = np.linalg.norm(b)
        if nb == 0:
            assert np.all(a == 0), name
            continue
        assert np.linalg.norm(a - b) / nb < 1e-2, (n, name)
    loss2, g2 = m.grad(Xd, Td)
    assert loss2 == loss and np.array_equal(g, g2)
