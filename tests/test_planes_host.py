"""One plane of a cell on its own (hyq_planes.h, what a lane of the planes kernel does) against
the one-cell form: the same Jacobian entries, decisions, extremes and flags, bit for bit, on
the host build."""
import numpy as np
import pytest

import cellhost as C
from _common import gaussian_raw, mixture_raw, to35


def cells(seed, n=120):
    """Mixtures (many with complex planes), near-Maxwellian cells (nearly double eigenvalues),
    and cells whose planes are not finite or not realizable."""
    rng = np.random.default_rng(seed)
    out = [to35(mixture_raw(rng, spread=1.5, lam_lo=0.01)) for _ in range(n)]
    for k in range(n // 2):
        M = to35(gaussian_raw(0.3 + rng.random(), rng.normal(size=3), np.eye(3) * 10.0 ** rng.uniform(-6, 1)))
        out.append(M * (1.0 + 1e-9 * rng.standard_normal(35) * (k % 2)))
    for v in (0.0, -1.0, np.nan, np.inf, 1e-300):
        for t in (0, 2, 9, 19, 34):
            M = out[t].copy()
            M[t] = v
            out.append(M)
    return out


@pytest.mark.parametrize("seed", range(3))
def test_plane_of_a_set_is_the_plane_of_the_cell(seed):
    for M in cells(seed):
        for q in range(5):
            a, b = C.plane_both(M, q)
            assert np.array_equal(a, b, equal_nan=True), (q, a, b)


@pytest.mark.parametrize("em", [0, 1])
@pytest.mark.parametrize("fin", [0, 1])
def test_decision_equals_the_one_cell_solve(em, fin):
    kinds = set()
    for M in cells(7 + em):
        for q in range(5):
            a, b = C.plane_decide(M, em, q, fin)
            assert np.array_equal(a, b, equal_nan=True), (q, a, b)
            kinds.add((bool(a[0]), bool(a[1])))
    assert (True, False) in kinds and (True, True) in kinds
