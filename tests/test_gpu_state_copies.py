"""States travel between host and device unchanged, whatever way a size and a memory kind take:
the runtime's copy (small, or pinned), or the ring of pinned chunks (8 MiB and more), with
whole and partial last chunks."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 29952 cells: 8386560 B, below 8 MiB; then 9 chunks of 1 MiB, 16 of 2 MiB, 17 and 29 of 4 MiB (the
# ring holds 10; from 64 MiB on the way up takes it too); the last chunk is a partial one
@pytest.mark.parametrize("N", [(1, 1, 1), (32, 26, 36), (32, 32, 30), (61, 53, 37), (67, 61, 59), (79, 75, 71)])
def test_round_trip(N):
    import torch
    import hyqmom_amd as H
    from hyqmom_amd.ensemble import jets_params
    rng = np.random.default_rng(sum(N))
    s = H.Solver(jets_params(N, 1.5, 0.01, "fp64"))
    for k in range(3):
        M = np.asfortranarray(rng.standard_normal(N + (35,)))
        s.set_state(M)
        assert np.array_equal(s.get_state(), M)
    pinned = torch.empty(M.size, dtype=torch.float64, pin_memory=True).numpy()
    pinned[:] = M.ravel(order="F")[::-1]
    P = pinned.reshape(M.shape, order="F")
    s.set_state(P)
    assert np.array_equal(s.get_state(), P)
    s.close()


def test_two_threads_read_one_state():
    import hyqmom_amd as H
    from hyqmom_amd.ensemble import jets_params
    N = (64, 60, 33)
    M = np.asfortranarray(np.random.default_rng(3).standard_normal(N + (35,)))
    s = H.Solver(jets_params(N, 1.5, 0.01, "mixed"))
    s.set_state(M)
    out = [None, None]

    def read(i):
        out[i] = s.get_state()

    t = [threading.Thread(target=read, args=(i,)) for i in range(2)]
    [x.start() for x in t]
    [x.join() for x in t]
    assert np.array_equal(out[0], M) and np.array_equal(out[1], M)
    s.close()


def test_ensemble_round_trip():
    """Runs of one cell, odd sizes and 8 MiB and more, set in any order; a set state leaves the
    other runs alone and starts its run over."""
    from hyqmom_amd.ensemble import Ensemble, jets_params
    sizes = [(1, 1, 1), (7, 5, 3), (37, 31, 29), (16, 16, 1), (64, 33, 32)]
    rng = np.random.default_rng(9)
    e = Ensemble([jets_params(N, 1.0, 0.1, "mixed") for N in sizes])
    S = [np.asfortranarray(rng.standard_normal(N + (35,))) for N in sizes]
    for r in (3, 0, 4, 2, 1):
        e.set_state(r, S[r])
    for r in range(len(S)):
        assert np.array_equal(e.get_state(r), S[r])
    from hyqmom_amd import initial_state
    e.set_initial_states()
    e.run(2)
    other = e.get_state(2)
    assert list(e.status()[2]) == [2] * len(S)
    e.set_state(4, S[4])
    assert list(e.status()[2]) == [2, 2, 2, 2, 0]
    assert np.array_equal(e.get_state(4), S[4]) and np.array_equal(e.get_state(2), other)
    e.close()
