"""k_hard's forms by the length of its list: up to 65536 entries, and (FP64 and mixed modes) the
form of two waves per SIMD beyond, in one turn and more; short and long lists of final solves
(fast mode).  Every cell's result is the same bits whatever the list around it."""
import numpy as np
import pytest

from test_gpu_fast_batch import HYQ_PREC_FP64, HYQ_PREC_MIXED_NEWTON, batch, mixed_cells

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hard():
    """Cells with an eigenvalue correction and finite results: each is an entry of the list."""
    from hyqmom_amd import _lib as L
    M = mixed_cells()
    Mr, F, vp, fl = batch(L.lib().hyq_wavespeed_batch, M, HYQ_PREC_FP64)
    M = M[((fl & 0x1C0) != 0) & np.isfinite(vp).all(axis=0) & np.isfinite(F).all(axis=0)]
    assert len(M) > 500
    return M, {p: batch(L.lib().hyq_wavespeed_batch, M, p) for p in (HYQ_PREC_FP64, HYQ_PREC_MIXED_NEWTON)}


# per block: 1; 2; 16 entries; just above half a block's threads; a full block; more than all blocks hold at
# one wave per SIMD; and at two
@pytest.mark.parametrize("n", [200, 512, 4096, 33000, 65536, 65537, 131073])
@pytest.mark.parametrize("precision", [HYQ_PREC_FP64, HYQ_PREC_MIXED_NEWTON])
def test_batches_of_entries(hard, n, precision):
    from hyqmom_amd import _lib as L
    M, want = hard
    idx = (np.arange(n, dtype=np.int64) * 7 + 3) % len(M)
    got = batch(L.lib().hyq_wavespeed_batch, M[idx], precision)
    for w, g in zip(want[precision], got):
        assert np.array_equal(w[..., idx], g, equal_nan=True)


@pytest.mark.parametrize("precision", ["fp64", "mixed", "mixed_newton", "mixed_learned"])
def test_steps_whose_cells_are_all_entries(hard, precision):
    """One step from a state without variation in z (then Mz = M exactly), at 4920, 67240 (planes
    spread over waves) and 98400 cells (planes in turn)."""
    import hyqmom_amd as H
    from hyqmom_amd.ensemble import jets_params
    M, _ = hard
    plane = M[(np.arange(41 * 40) * 7 + 3) % len(M)].reshape(41, 40, 1, 35)
    out = {}
    for Nz in (3, 41, 60):
        p = dict(jets_params((41, 40, Nz), 1.5, 0.01, precision), dtmax=1e-7)
        s = H.Solver(p)
        s.set_state(np.asfortranarray(np.repeat(plane, Nz, axis=2)))
        s.step()
        out[Nz] = s.get_state()
        s.close()
        assert np.array_equal(out[Nz], np.repeat(out[Nz][:, :, :1, :], Nz, axis=2))
    assert not np.array_equal(out[3][:, :, 0, :], plane[:, :, 0, :])
    for Nz in (41, 60):
        assert np.array_equal(out[3][:, :, 0, :], out[Nz][:, :, 0, :]), Nz
