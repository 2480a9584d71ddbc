"""Edges of the dispatch rules and of the kernels' tiles: sizes around the
limits at which a kernel variant takes over or a tile is partly filled.

Bars: FP64 results are the oracle's (or another route's) bit for bit; FP32
block products within their rounding."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
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


def _oracle_iterates(pr, stop, iters):
    """x after `iters` iterations of the oracle in the device's order."""
    gc = pr.g_coord()
    K = (O.assemble_elastic(gc, pr.e, pr.v, pr.e_elem, nthreads=8) if pr.kind == "elastic"
         else O.assemble_laplace(gc, pr.kx, pr.ky, pr.kz, pr.k_elem, nthreads=8))
    dg = O.diag(pr.g_g, K, pr.neq)
    kw = {}
    r = pr.r0.copy()
    if pr.fix_eq is not None:
        store = dg[pr.fix_eq - 1] + P.PENALTY
        dg[pr.fix_eq - 1] = store
        r[pr.fix_eq - 1] = store * pr.fix_val
        kw = {"no_f": pr.fix_eq, "store": store}
    return O.pcg(pr.g_g, K, r, dg, 0.0, iters, stop=O.STOP_CHECON if stop == "checon" else O.STOP_RELRES,
                 dot_order=O.DOT_DEVICE, nthreads=8, **kw)[0]


# Reduction blocks (256 equations) at the edges of the rules: one; 512 | 513
# (p formed in the products | not); 2,048 | 2,049 (no fold launches | folds)
@pytest.mark.parametrize("box", [(5, 5, 5), (31, 63, 63), (32, 63, 63), (63, 63, 127), (64, 63, 127)])
@pytest.mark.parametrize("stop", ["checon", "relres"])
def test_iteration_tiers_bitexact(box, stop):
    pr = P.laplace_cube(1, nels_xyz=box)
    print(f"[gpu-test] tiers {box} neq={pr.neq} {stop}", flush=True)
    with Context(0) as ctx:
        r = P.setup(ctx, pr)
        ctx.pcg_begin(r, 7, 0.0, stop=stop)
        ctx.pcg_run(3)          # p is complete between runs
        ctx.pcg_run(1)
        ctx.pcg_run(5)          # three iterations to the limit, then nothing
        assert ctx.pcg_poll().iters == 7
        assert np.array_equal(ctx.pcg_x(), _oracle_iterates(pr, stop, 7))


def test_more_slots_than_the_padded_table_holds():
    """Equations that more than eight elements list (freedoms tied together)
    take the iteration that reads the slot list itself: the oracle's bits."""
    pr = P.elastic_cube(3)
    g = pr.g_g.copy()
    # the z freedoms of the top face become one equation
    top = np.nonzero(np.abs(pr.mesh.coords[:, 2]) < 1e-12)[0]
    tied = pr.nf[top, 2]
    g[np.isin(g, tied)] = tied[0]
    keep = np.unique(g[g > 0])
    new = np.zeros(pr.neq + 1, dtype=np.int32)
    new[keep] = np.arange(1, keep.size + 1)
    r = np.zeros(keep.size)
    np.add.at(r, new[np.where(np.isin(np.arange(1, pr.neq + 1), tied), tied[0], np.arange(1, pr.neq + 1))] - 1, pr.r0)
    tp = P.Problem("elastic", pr.mesh, new[g], keep.size, r, pr.nf, e=pr.e, v=pr.v)
    assert np.bincount(tp.g_g.ravel())[1:].max() > 8
    with Context(0) as ctx:
        P.setup(ctx, tp)
        x, res = ctx.pcg_solve(r, 40, 0.0, stop="relres")
        assert res.iters == 40 and np.array_equal(x, _oracle_iterates(tp, "relres", 40))
