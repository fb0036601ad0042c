"""Both shapes of the FP64 plane solves around the line between them, 1024 blocks of 64 cells: every
cell's result is the same bits."""
import numpy as np
import pytest

from test_gpu_fast_batch import HYQ_PREC_FP64, batch, mixed_cells

pytestmark = pytest.mark.gpu


def test_fp64_batches_around_the_line():
    from hyqmom_amd import _lib as L
    M = mixed_cells()
    fn = L.lib().hyq_wavespeed_batch
    want = batch(fn, M, HYQ_PREC_FP64)
    for n in (65472, 65473):  # 1023 blocks; 1024
        idx = (np.arange(n, dtype=np.int64) * 4099 + 7) % len(M)
        for w, g in zip(want, batch(fn, M[idx], HYQ_PREC_FP64)):
            assert np.array_equal(w[..., idx], g, equal_nan=True)
