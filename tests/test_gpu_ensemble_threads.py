"""The first calls of a new ensemble, and several host threads on one: each sets and reads its own run while the others do the
same (the calls share one staging buffer on the device), and reads a state while steps run."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _together(fns):
    errors = []

    def guard(f):
        try:
            f()
        except Exception as e:  # an assertion of another thread fails the test too
            errors.append(e)

    t = [threading.Thread(target=guard, args=(f,)) for f in fns]
    [x.start() for x in t]
    [x.join() for x in t]
    if errors:
        raise errors[0]


# one copy each; through the ring down (8 MiB and more); through the ring both ways (64 MiB and more)
@pytest.mark.parametrize("sizes", [[(7, 5, 3), (13, 11, 7), (5, 5, 1), (1, 1, 1)],
                                   [(33, 32, 30), (32, 31, 33)],
                                   [(64, 64, 60), (61, 65, 62)]])
def test_threads_on_their_own_runs(sizes):
    from hyqmom_amd.ensemble import Ensemble, jets_params
    e = Ensemble([jets_params(N, 1.0, 0.1, "mixed") for N in sizes])

    def work(r):
        def f():
            rng = np.random.default_rng(r)
            for k in range(6):
                M = np.asfortranarray(rng.standard_normal(sizes[r] + (35,)))
                e.set_state(r, M)
                for _ in range(3):
                    assert np.array_equal(e.get_state(r), M), (r, k)
        return f

    _together([work(r) for r in range(len(sizes))])
    e.close()


def test_the_first_calls_of_a_new_ensemble():
    """A new ensemble's state is zero, and a state set at once stays (the fill at creation is done
    before either): 61 MB of planes, an upload of one cell."""
    from hyqmom_amd.ensemble import Ensemble, jets_params
    one = np.arange(1.0, 36.0).reshape(1, 1, 1, 35)
    for k in range(4):
        e = Ensemble([jets_params((1, 1, 1), 1.0, 0.1, "mixed"), jets_params((60, 60, 60), 1.0, 0.1, "mixed")])
        e.set_state(0, one)
        assert np.array_equal(e.get_state(0), one)
        assert not e.get_state(1).any()
        e.close()


def test_a_state_read_while_steps_run():
    """Every read gives a state that the run had between two calls of run()."""
    from hyqmom_amd import initial_state
    from hyqmom_amd.ensemble import Ensemble, jets_params
    runs = [jets_params((20, 20, 10), 1.0, 0.5, "fp64"), jets_params((17, 13, 11), 0.7, 0.3, "fp64")]
    for p in runs:
        p["CFL"] = 0.2
    e = Ensemble(runs)

    def start():
        for r, p in enumerate(runs):
            e.set_state(r, initial_state(p))

    start()
    had = [e.get_state(1).tobytes()]
    for _ in range(8):
        e.run(1)
        had.append(e.get_state(1).tobytes())
    start()
    read = []
    _together([lambda: [e.run(1) for _ in range(8)],
               lambda: [read.append(e.get_state(1).tobytes()) for _ in range(40)]])
    assert all(s in had for s in read)
    e.close()
