"""The forms of the step's kernels that a size selects, against one another: every cell's result
is the same bits whatever the batch or grid around it.  (The values themselves are held
against the oracle by the parity, golden-run and batch tests.)"""
import numpy as np
import pytest

from test_gpu_fast_batch import HYQ_PREC_FP64, HYQ_PREC_MIXED_NEWTON, batch, mixed_cells

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def base():
    """9912 cells: jets (near-Maxwellian) and stress cells (complex planes, z re-projections),
    and their results in one batch of each precision."""
    from hyqmom_amd import _lib as L
    M = mixed_cells()
    fn = L.lib().hyq_wavespeed_batch
    return M, {p: batch(fn, M, p) for p in (HYQ_PREC_FP64, HYQ_PREC_MIXED_NEWTON)}


# one cell; around a wave; an odd count; around the 1280 blocks from which a wave takes all
# planes of its cells; around the 200000 cells from which every phase is a launch of its own
@pytest.mark.parametrize("n", [1, 63, 65, 4099, 81856, 81857, 199999, 200001])
@pytest.mark.parametrize("precision", [HYQ_PREC_FP64, HYQ_PREC_MIXED_NEWTON])
def test_a_cell_does_not_depend_on_its_batch(base, n, precision):
    from hyqmom_amd import _lib as L
    M, want = base
    # a stride that is coprime with the count mixes the two kinds of cells in every wave
    idx = (np.arange(n, dtype=np.int64) * 4099 + 7) % len(M)
    got = batch(L.lib().hyq_wavespeed_batch, M[idx], precision)
    for w, g in zip(want[precision], got):
        assert np.array_equal(w[..., idx], g, equal_nan=True)


def test_a_batch_of_hard_cells_only(base):
    """Every cell on the correction path, and none: lists of full and of zero length."""
    from hyqmom_amd import _lib as L
    M, want = base
    fl = want[HYQ_PREC_FP64][3]
    hard = np.nonzero(fl & 0xFF0)[0]
    easy = np.nonzero((fl & 0xFFF) == 0)[0]
    assert len(hard) > 100 and len(easy) > 100
    for sel in (hard, easy):
        idx = np.resize(sel, 5001)
        for p in (HYQ_PREC_FP64, HYQ_PREC_MIXED_NEWTON):
            got = batch(L.lib().hyq_wavespeed_batch, M[idx], p)
            for w, g in zip(want[p], got):
                assert np.array_equal(w[..., idx], g, equal_nan=True)


def test_batch_in_place_and_without_flags(base):
    """Mr may be M itself, and the FP64 batch runs without the flags output."""
    from gpu_util import empty_dev, to_dev, to_host
    from hyqmom_amd import _lib as L
    M, want = base
    n = 777
    Mr, F, vp = to_dev(np.ascontiguousarray(M[:n].T)), empty_dev((105, n)), empty_dev((6, n))
    p = F.data_ptr()
    L.check(L.lib().hyq_wavespeed_batch(Mr.data_ptr(), n, 1.5, 0, 1, HYQ_PREC_FP64, Mr.data_ptr(), p,
                                        p + 35 * n * 8, p + 70 * n * 8, vp.data_ptr(), None), "batch")
    for w, g in zip(want[HYQ_PREC_FP64], (Mr, F, vp)):
        assert np.array_equal(w[..., :n], to_host(g), equal_nan=True)


@pytest.mark.parametrize("precision", [HYQ_PREC_FP64, HYQ_PREC_MIXED_NEWTON])
def test_moments_at_the_underflow_scale(precision):
    """A cell at the front of a spreading jet (120x120x60, step 19): a Maxwellian of rho = 0.1 but
    for moments of 1e-26 to 1e-86, whose QR bulges have subnormal squares.  Its speeds are the
    Maxwellian's, +- sqrt(6) from the 1D closure; the deviations are below 1e-24."""
    from hyqmom_amd import _lib as L
    cell = np.array([1e-01, -1.57268323e-26, 1e-01, -4.70059143e-26, 3e-01, 1.34347720e-43, 3.29407251e-26,
                     5.31150428e-43, 9.86852473e-26, 1e-01, -8.22074091e-26, 1e-01, 5.35310728e-43,
                     1.78791113e-25, 3e-01, 0.0, -3.98547105e-44, -6.44043138e-63, -1.02113400e-43, 1e-01,
                     -1.62554612e-26, 1e-01, 0.0, -2.26151976e-43, 3e-01, 0.0, -5.35438946e-86, 6.44062650e-63,
                     0.0, -1.70396464e-43, 0.0, 1.34347720e-43, 3.34254778e-26, 0.0, 1e-01])
    got = batch(L.lib().hyq_wavespeed_batch, np.stack([cell] * 3), precision)
    want = np.sqrt(6.0) * np.array([-1.0, 1.0] * 3)[:, None]
    assert np.abs(got[2] - want).max() < 1e-12
    assert np.isfinite(got[1]).all()


@pytest.mark.parametrize("precision", ["fp64", "mixed", "mixed_newton"])
def test_step_forms_agree(precision):
    """A state without variation in z is the same in every plane of any depth; the depths lie
    below and above the grids from which a thread updates all moments of a cell (65536 cells)
    and a wave takes all planes of its cells (pass 1 81920; pass 2 131072, FP64 262144).  Zero gradient in z:
    Mz = M exactly.  dt is fixed by dtmax."""
    import hyqmom_amd as H
    from hyqmom_amd.ensemble import jets_params
    p0 = jets_params((41, 39, 4), 1.5, 0.01, precision)
    p0["dtmax"] = 1e-4
    M0 = H.initial_state(p0)[:, :, 2:3, :]
    out = {}
    for Nz in (3, 40, 41, 51, 52, 81, 83, 163, 165):  # 1599 cells a plane
        p = dict(p0, Nz=Nz)
        s = H.Solver(p)
        s.set_state(np.asfortranarray(np.repeat(M0, Nz, axis=2)))
        s.run(10.0, 4)
        M = s.get_state()
        s.close()
        assert np.array_equal(M, np.repeat(M[:, :, :1, :], Nz, axis=2))
        out[Nz] = M[:, :, 0, :]
    assert not np.array_equal(out[3], M0[:, :, 0, :])
    for Nz in out:
        assert np.array_equal(out[3], out[Nz]), Nz


@pytest.mark.parametrize("precision", ["fp64", "mixed", "mixed_newton"])
def test_a_run_does_not_depend_on_its_ensemble(precision):
    """93k cells in all, more than the 81920 from which a wave takes all planes of its cells; each
    run on its own is below.  Odd grids, one of a single plane, and one that has ended."""
    from hyqmom_amd import initial_state
    from hyqmom_amd.ensemble import Ensemble, jets_params
    runs = [jets_params((37, 31, 29), 1.5, 0.01, precision), jets_params((16, 17, 1), 0.7, 0.3, precision),
            jets_params((41, 33, 33), 0.9, 0.05, precision), jets_params((25, 24, 24), 1.2, 1.0, precision)]
    runs[3]["tmax"] = 0.004  # ends within the steps

    def run(ps):
        e = Ensemble(ps)
        for r, p in enumerate(ps):
            e.set_state(r, initial_state(p))
        e.run(5)
        out = [e.get_state(r) for r in range(len(ps))], e.status()
        e.close()
        return out

    M, (t, dt, nn) = run(runs)
    assert nn[3] < 5
    for r, p in enumerate(runs):
        (m,), (t1, dt1, nn1) = run([p])
        assert np.array_equal(M[r], m, equal_nan=True), r
        assert (t[r], dt[r], nn[r]) == (t1[0], dt1[0], nn1[0])
