"""Edges of the dispatch rules and of the kernels' tiles: sizes around the
limits at which a kernel variant takes over or a tile is partly filled.

Bars: FP64 results are the oracle's (or another route's) bit for bit; FP32
block products within their rounding."""
import ctypes as C

import numpy as np
import pytest

from parafem_amd import Context, problems as P
from parafem_amd.api import BlockOpts, BlockResult, lib

pytestmark = pytest.mark.gpu


# Block partials folded: 3 and 5 (parts with none, or one more than others),
# 23, 103, and 2,048 (the cap: the serial chains at their longest).  One block
# iteration gives x = (r,d)/(p,Kp) p with p = d = dinv r; a dropped or doubled
# partial moves it by at least 1/2,048.  Bar 1e-4: FP32 products of 60 terms
# round to about 60 * 2^-24 = 4e-6 of their largest partial sum, and the sums
# of Kp over 8 elements cancel by a factor of ten or so.
@pytest.mark.parametrize("box", [(1, 1, 1), (1, 1, 2), (2, 3, 4), (5, 5, 5), (22, 22, 22)])
def test_block_fold_sizes(box):
    pr = P.elastic_cube(1, lognormal_e=True, nels_xyz=box)
    print(f"[gpu-test] block folds {box} neq={pr.neq}", flush=True)
    rng = np.random.default_rng(5)
    F = np.asfortranarray(np.stack([pr.r0, rng.standard_normal(pr.neq), rng.standard_normal(pr.neq)], axis=1))
    X = np.zeros(F.shape, order="F")
    with Context(0) as ctx:
        P.setup(ctx, pr)
        pd = C.POINTER(C.c_double)
        o, res = BlockOpts(1e-10, 0.0, 1, 0, 1), BlockResult()      # one iteration
        lib().pf_block_solve(ctx.h, 3, F.ctypes.data_as(pd), X.ctypes.data_as(pd), C.byref(o), C.byref(res))
        assert res.inner_iters == 1
        dinv = 1.0 / ctx.diag_get()
        for c in range(3):
            p = dinv * F[:, c]
            x = (F[:, c] @ p) / (p @ ctx.apply(p)) * p
            assert np.abs(X[:, c] - x).max() <= 1e-4 * np.abs(x).max()
