"""A state read many times comes back unchanged each time: the first reads of an object go through
the runtime, later ones (after 13 at 9 MB, 4 at 16, two at 24) through the ring of pinned chunks;
and from several threads across the change."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [(32, 32, 30), (40, 40, 36), (45, 44, 43), (47, 46, 41), (61, 53, 37), (56, 56, 55), (60, 60, 57), (61, 60, 59)])
def test_repeated_reads(N):
    import hyqmom_amd as H
    from hyqmom_amd.ensemble import jets_params
    rng = np.random.default_rng(sum(N))
    s = H.Solver(jets_params(N, 1.5, 0.01, "mixed"))
    for k in range(20):
        M = np.asfortranarray(rng.standard_normal(N + (35,)))
        s.set_state(M)
        assert np.array_equal(s.get_state(), M), k
    s.close()


def test_threads_across_the_change():
    import hyqmom_amd as H
    from hyqmom_amd.ensemble import jets_params
    N = (40, 40, 36)
    M = np.asfortranarray(np.random.default_rng(4).standard_normal(N + (35,)))
    s = H.Solver(jets_params(N, 1.5, 0.01, "mixed"))
    s.set_state(M)
    same = []

    def read():
        for _ in range(6):
            same.append(np.array_equal(s.get_state(), M))

    t = [threading.Thread(target=read) for _ in range(3)]
    [x.start() for x in t]
    [x.join() for x in t]
    assert len(same) == 18 and all(same)
    s.close()
