"""closure_and_eigenvalues where the density or the variance is at the end of FP64's range: IEEE
quotients of such numbers are finite, and so are the speeds."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sets():
    """Moment sets whose recurrence is exact in FP64 at every scale, with their speeds: a Gaussian
    with mean 0 or 1 (speeds u +- sqrt(6)) at densities down to the smallest numbers, and density
    1 with a variance s and fourth moment s / 2 (b2 = s, b3 = 1/2: speeds +- sqrt(s + 5/4))."""
    out = []
    for e in (0, -500, -899, -901, -1000, -1020, -1022, -1023, -1025, -1030, -1050, -1070):
        s = 2.0 ** e
        out.append(([s, 0.0, s, 0.0, 3 * s], -np.sqrt(6.0), np.sqrt(6.0)))
        out.append(([s, s, 2 * s, 4 * s, 10 * s], 1 - np.sqrt(6.0), 1 + np.sqrt(6.0)))
        if e <= -500:
            out.append(([1.0, 0.0, s, 0.0, s / 2], -np.sqrt(1.25), np.sqrt(1.25)))
    return out


def test_small_densities_and_variances():
    from gpu_util import empty_dev, to_dev, to_host
    from hyqmom_amd import _lib as L
    sets = _sets()
    n = len(sets)
    m = to_dev(np.ascontiguousarray(np.array([s[0] for s in sets]).T))
    lo, hi = empty_dev((n,)), empty_dev((n,))
    L.check(L.lib().hyq_closure1d_batch(m.data_ptr(), n, lo.data_ptr(), hi.data_ptr()), "closure1d")
    # the roots come from acos and cos of FP64: a few units in the last place of 3.5
    assert np.abs(to_host(lo) - [s[1] for s in sets]).max() < 1e-14
    assert np.abs(to_host(hi) - [s[2] for s in sets]).max() < 1e-14
