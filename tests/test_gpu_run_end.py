"""Runs that end at tmax in one call, whatever number of steps the call queues at a time, against
the same steps taken one by one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = (21, 19, 10)


def params(tmax, precision="fp64"):
    from hyqmom_amd.ensemble import jets_params
    p = jets_params(N, 0.7, 0.5, precision)
    p.update(CFL=0.2, dtmax=1e-5, tmax=tmax)
    return p


# steps to the end (dt is dtmax, the last step shorter): within the first piece, around it, in the
# second, and past a whole chunk
@pytest.mark.parametrize("steps", [1, 3, 15, 16, 17, 40, 83])
@pytest.mark.parametrize("nnmax", [10 ** 9, 81])
def test_run_to_tmax(steps, nnmax):
    import hyqmom_amd as H
    tmax = (steps - 0.5) * 1e-5
    p = params(tmax)
    a, b = H.Solver(p), H.Solver(p)
    M0 = H.initial_state(p)
    a.set_state(M0)
    b.set_state(M0)
    a.run(tmax, nnmax)
    while b.t < tmax and b.nn < nnmax:
        b.step()
    assert a.nn == b.nn == min(steps, nnmax) and a.t == b.t
    assert np.array_equal(a.get_state(), b.get_state())
    a.run(tmax, a.nn + 5)  # nothing is left to do, or five steps more
    for _ in range(5):
        if b.t < tmax:
            b.step()
    assert (a.nn, a.t) == (b.nn, b.t) and np.array_equal(a.get_state(), b.get_state())
    a.close()
    b.close()


@pytest.mark.parametrize("graph", [True, False])
def test_ensemble_runs_end_at_their_own_tmax(graph):
    from hyqmom_amd import initial_state
    from hyqmom_amd.ensemble import Ensemble
    runs = [params((k - 0.5) * 1e-5, "mixed") for k in (3, 8, 9, 30)]
    a, b = Ensemble(runs), Ensemble(runs)
    for r, p in enumerate(runs):
        a.set_state(r, initial_state(p))
        b.set_state(r, initial_state(p))
    a.run(0, graph=graph)
    for n in (7, 2, 500, 1):
        a.run(n, graph=graph)
    for _ in range(31):
        b.run(1)
    sa, sb = a.status(), b.status()
    assert list(sa[2]) == [3, 8, 9, 30]
    for x, y in zip(sa, sb):
        assert np.array_equal(x, y)
    for r in range(len(runs)):
        assert np.array_equal(a.get_state(r), b.get_state(r))
    a.set_state(1, initial_state(runs[1]))  # one run starts over, alone
    a.run(50, graph=graph)
    assert list(a.status()[2]) == [3, 8, 9, 30] and np.array_equal(a.get_state(1), b.get_state(1))
    a.close()
    b.close()
