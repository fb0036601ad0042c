"""The two forms of the realizability projection, hyq_closure_batch's (every 4x4 minor's cubic
inlined) and the step kernels' (one copy in a loop), against one another."""
import numpy as np
import pytest

from test_gpu_fast_batch import HYQ_PREC_FP64, batch, mixed_cells

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 127, 129, 9912])
def test_closure_batch_has_the_bits_of_the_wave_speed_batch(n):
    """Cells that no eigenvalue correction and no z path touches: the wave-speed batch gives the
    closure and fluxes of their projected state.  (The flags of the second projection are
    ORed to the first's there.)"""
    from gpu_util import empty_dev, to_dev, to_host
    from hyqmom_amd import _lib as L
    M = mixed_cells()
    M = M[(np.arange(n) * 4099 + 7) % len(M)]
    want = batch(L.lib().hyq_wavespeed_batch, M, HYQ_PREC_FP64)
    plain = (want[3] & 0xFC0) == 0  # EIGCORR_X, _Y, _Z, ZNEGVAR, NONFINITE, RHOCLAMP
    A, Mr, F = empty_dev((35, n)), empty_dev((35, n)), empty_dev((105, n))
    fa, fb = empty_dev((n,), "int32"), empty_dev((n,), "int32")
    Md = to_dev(np.ascontiguousarray(M.T))
    p = F.data_ptr()
    # the projection without fluxes, then the closure of the projected state with them
    L.check(L.lib().hyq_closure_batch(Md.data_ptr(), n, 1.5, 0, A.data_ptr(), None, None, None, fa.data_ptr()), "closure")
    L.check(L.lib().hyq_closure_batch(A.data_ptr(), n, 1.5, 0, Mr.data_ptr(), p, p + 35 * n * 8, p + 70 * n * 8,
                                      fb.data_ptr()), "closure")
    got_flags = (to_host(fa) | to_host(fb)) & 0x3F
    if n > 1000:
        assert plain.sum() > n // 4 and (want[3][plain] & 0x3F).any()
        assert (got_flags[plain] & 0x20).any()  # ROOTS4: the cubics ran
    assert np.array_equal(to_host(Mr)[:, plain], want[0][:, plain], equal_nan=True)
    assert np.array_equal(to_host(F)[:, plain], want[1][:, plain], equal_nan=True)
    assert np.array_equal(got_flags[plain], want[3][plain] & 0x3F)
