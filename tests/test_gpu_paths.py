"""Edges of the dispatch rules and of the kernels' tiles: sizes around the
limits at which a kernel variant takes over or a tile is partly filled.

Bars: FP64 results are the oracle's (or another route's) bit for bit; FP32
block products within their rounding."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from parafem_amd import Batch, Context, DeviceArray, mesh as M, problems as P
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


def _mesh_problem(ntot, box):
    if ntot == 60:
        return P.elastic_cube(1, nels_xyz=box, lognormal_e=True)
    if ntot == 8:
        pr = P.laplace_cube(1, nels_xyz=box)
        pr.fix_eq = pr.fix_val = None
        return pr
    m = M.box_hex8(*box)
    nf, neq = M.steering(m.nn, 3, M.base_fixed_rest(m))
    r = np.random.default_rng(1).standard_normal(neq)
    return P.Problem("elastic", m, M.g_g_from(nf, m.g_num), neq, r, nf)


def _matrices(kind, nels, nt, seed=3):
    """Element matrices (element, column, row): symmetric but for the rounding
    the packed triangle keeps ("ulps"), exactly symmetric, with one
    difference of more bits than it keeps in the last element ("wide"),
    without symmetry, or with a whole range of magnitudes ("ranges")."""
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((nels, nt, nt))
    if kind == "general":
        return a
    K = np.matmul(a, a.transpose(0, 2, 1)) + nt * np.eye(nt)
    K = (K + K.transpose(0, 2, 1)) / 2
    if kind == "ranges":
        d = 2.0 ** rng.integers(-300, 300, (nels, 1, 1))
        K = K * d
    low = np.tril(np.ones((nt, nt), dtype=bool), -1)
    if kind != "symmetric":
        K[:, low] += np.ldexp(rng.integers(-900, 900, (nels, low.sum())), -48 + np.frexp(np.abs(K).max((1, 2)))[1][:, None] - 6)
    if kind == "wide":
        K[-1, 3, 1] = K[-1, 1, 3] * (1 + 2.0 ** -12 + 2.0 ** -40)
    return K


# FP64 matrices as the packed triangle (the first three kinds, above 32 MB) and
# whole (the others, and all kinds up to 32 MB): entries, products and iterates
# bit for bit.  Element counts around the lane groups: 16 elements a wavefront
# for ntot 8 (65,545 = 16 * 4,096 + 9 and 65,551), 2 for 24, 1 for 60.
@pytest.mark.parametrize("ntot,box", [(60, (3, 1, 2)), (60, (11, 11, 10)), (24, (3, 3, 1)), (24, (20, 19, 20)),
                                      (24, (23, 317, 1)), (8, (5, 3, 1)), (8, (5, 13109, 1)), (8, (65551, 1, 1)),
                                      (8, (41, 40, 40))])
@pytest.mark.parametrize("kind", ["ulps", "symmetric", "ranges", "wide", "general"])
def test_fp64_storage_bitexact(ntot, box, kind):
    pr = _mesh_problem(ntot, box)
    print(f"[gpu-test] fp64 storage {ntot} {box} {kind}", flush=True)
    K = _matrices(kind, pr.nels, ntot)
    rng = np.random.default_rng(7)
    with Context(0) as ctx:
        ctx.mesh_set(pr.g_coord())
        ctx.steer_set(pr.g_g, pr.neq)
        before = ctx.mem_used()
        ctx.storkm_set(K)
        if pr.nels * ntot * ntot * 8 > 32 << 20 and kind in ("ulps", "symmetric", "ranges"):
            # the triangle (without the kept staging buffer): less than whole matrices
            ctx.trim()
            assert ctx.mem_used() - before < 0.8 * pr.nels * ntot * ntot * 8
        assert np.array_equal(ctx.storkm_get(), K)
        assert np.array_equal(ctx.diag_get(), O.diag(pr.g_g, K, pr.neq))
        x = rng.standard_normal(pr.neq)
        assert np.array_equal(ctx.apply(x), O.apply(pr.g_g, K, x))
        pm = rng.standard_normal((pr.nels, ntot))
        d, u = DeviceArray.from_host(ctx, pm), DeviceArray(ctx, pm.size)
        ctx.elem_matvec(d, u)
        assert np.array_equal(u.download().reshape(pm.shape), O.elem_matvec(K, pm))
        if kind in ("ulps", "symmetric"):      # positive definite: whole iterations
            dg = O.diag(pr.g_g, K, pr.neq)
            r = rng.standard_normal(pr.neq)
            xg, res = ctx.pcg_solve(r, 5, 0.0, stop="relres")
            xo = O.pcg(pr.g_g, K, r, dg, 0.0, 5, stop=O.STOP_RELRES, dot_order=O.DOT_DEVICE)[0]
            assert np.array_equal(xg, xo)


# Zeros with a sign: equal ones on both sides of the diagonal, one only above or
# only below it (which the triangle cannot tell, so the matrices stay whole).
@pytest.mark.parametrize("ntot,box", [(60, (11, 11, 10)), (24, (20, 19, 20)), (8, (41, 40, 40))])
@pytest.mark.parametrize("where", ["both", "above", "below"])
def test_fp64_storage_keeps_the_sign_of_zeros(ntot, box, where):
    pr = _mesh_problem(ntot, box)
    K = _matrices("ulps", pr.nels, ntot)
    for a, b in ((0, 2), (1, 5), (3, 7), (4, ntot - 1)):        # K[e, column, row]
        K[:, a, b] = -0.0 if where in ("both", "below") else 0.0
        K[:, b, a] = -0.0 if where in ("both", "above") else 0.0
    print(f"[gpu-test] signed zeros {ntot} {where}", flush=True)
    with Context(0) as ctx:
        ctx.mesh_set(pr.g_coord())
        ctx.steer_set(pr.g_g, pr.neq)
        before = ctx.mem_used()
        ctx.storkm_set(K)
        ctx.trim()
        packed = ctx.mem_used() - before < 0.8 * K.nbytes
        assert packed == (where != "below")
        assert np.array_equal(ctx.storkm_get().view(np.uint64), K.view(np.uint64))


def test_batch_of_whole_and_packed_matrices():
    """FP64 contexts that hold whole matrices and ones that hold the triangle
    advance in one batch, each as alone."""
    pr = P.elastic_cube(1, nels_xyz=(11, 11, 10))
    Ks = [_matrices(k, pr.nels, 60, seed) for k, seed in (("wide", 1), ("ulps", 2), ("symmetric", 3))]
    ctxs, ref = [], []
    for K in Ks:
        ctx = Context(0)
        ctx.mesh_set(pr.g_coord())
        ctx.steer_set(pr.g_g, pr.neq)
        ctx.storkm_set(K)
        ref.append(ctx.pcg_solve(pr.r0, 9, 0.0, stop="relres")[0])
        ctx.pcg_begin(pr.r0, 9, 0.0, stop="relres")
        ctxs.append(ctx)
    for persistent in (False, True):
        with Batch(0) as b:
            for ctx in ctxs:
                ctx.pcg_begin(pr.r0, 9, 0.0, stop="relres")
            b.run(ctxs, 12, persistent=persistent)
            for ctx, x in zip(ctxs, ref):
                ctx.sync()
                assert np.array_equal(ctx.pcg_x(), x)
    for ctx in ctxs:
        ctx.close()


# Matrices that the triangle cannot hold, seen in the first chunk of 128 MB or in
# the second one (after which the first one's are unpacked again): uploaded
# once, and no memory kept beyond whole matrices and a chunk.
@pytest.mark.parametrize("ntot,box", [(60, (11, 11, 10)), (60, (17, 17, 17)), (24, (31, 31, 31)), (8, (64, 64, 65))])
@pytest.mark.parametrize("kind", ["wide", "general"])
def test_upload_that_the_triangle_cannot_hold(ntot, box, kind):
    pr = _mesh_problem(ntot, box)
    chunk = (128 << 20) // (8 * ntot * ntot)
    print(f"[gpu-test] upload {ntot} {box} {kind} chunks {pr.nels / chunk:.2f}", flush=True)
    K = _matrices(kind, pr.nels, ntot)
    x = np.random.default_rng(3).standard_normal(pr.neq)
    with Context(0) as ctx:
        ctx.mesh_set(pr.g_coord())
        ctx.steer_set(pr.g_g, pr.neq)
        ctx.trim()
        before = ctx.mem_used()
        for _ in range(2):
            ctx.storkm_set(K)
            assert ctx.mem_used() - before <= K.nbytes + min(K.nbytes, 128 << 20) + (1 << 20)
        assert np.array_equal(ctx.storkm_get(), K)
        assert np.array_equal(ctx.diag_get(), O.diag(pr.g_g, K, pr.neq))
        assert np.array_equal(ctx.apply(x), O.apply(pr.g_g, K, x))
        ctx.storkm_set(np.ascontiguousarray((K + K.transpose(0, 2, 1)) / 2))     # and the triangle after it
        assert np.array_equal(ctx.storkm_get(), (K + K.transpose(0, 2, 1)) / 2)


# One batch of solves of every storage that a mesh's FP64 matrices can have, each
# storage's products a launch of their own over its own solves: storages first,
# last, between and alone in the batch.
@pytest.mark.parametrize("ntot,small,large", [(60, (5, 4, 3), (11, 11, 10)), (24, (7, 5, 4), (20, 19, 20)),
                                              (8, (9, 7, 5), (41, 40, 40))])
@pytest.mark.parametrize("order", ["wdWtD", "DtdwW", "dD", "wW", "t"])
def test_batch_of_every_storage(ntot, small, large, order):
    if ntot != 8:
        order = order.replace("t", "")
    if not order:
        pytest.skip("only 8 freedoms have triangles without differences")
    ctxs, prs, alone = [], [], []
    print(f"[gpu-test] batch storages {ntot} {order}", flush=True)
    for k, o in enumerate(order):
        pr = _mesh_problem(ntot, large if o in "dDW" else small)
        pr.r0 = np.random.default_rng(k).standard_normal(pr.neq)
        ctx = Context(0)
        if o == "t":            # assembled hex8 Laplace: the triangle without differences
            P.setup(ctx, pr)
        else:                   # w, W: whole (small; too wide a difference); d, D: with differences
            ctx.mesh_set(pr.g_coord())
            ctx.steer_set(pr.g_g, pr.neq)
            ctx.storkm_set(_matrices("wide" if o == "W" else "ulps", pr.nels, ntot, k))
        alone.append(ctx.pcg_solve(pr.r0, 9, 0.0, stop="relres")[0])
        ctxs.append(ctx)
        prs.append(pr)
    with Batch(0) as b:
        for kw in (dict(graph=True), dict(persistent=True), dict(graph=False), dict(graph=True)):
            for ctx, pr in zip(ctxs, prs):
                ctx.pcg_begin(pr.r0, 9, 0.0, stop="relres")
            b.run(ctxs, 5, **kw)
            b.run(ctxs, 5, **kw)
            for ctx, x in zip(ctxs, alone):
                assert ctx.pcg_poll().iters == 9 and np.array_equal(ctx.pcg_x(), x), kw
    for ctx in ctxs:
        ctx.close()


def test_one_large_solve_persistent_and_by_launches():
    """A single solve above 2,048 blocks, whose start lists and table are the
    same for the persistent kernel and for launches, but not its lists' lengths."""
    pr = P.laplace_cube(81)
    assert (pr.neq + 255) // 256 > 2048
    with Context(0) as ctx, Batch(0) as b:
        r = P.setup(ctx, pr)
        x = ctx.pcg_solve(r, 9, 0.0, stop="relres")[0]
        for kw in (dict(persistent=True), dict(graph=False), dict(persistent=True), dict(graph=True), dict(graph=False)):
            ctx.pcg_begin(r, 9, 0.0, stop="relres")
            b.run([ctx], 5, **kw)
            b.run([ctx], 5, **kw)
            assert ctx.pcg_poll().iters == 9 and np.array_equal(ctx.pcg_x(), x), kw


def test_assembly_that_the_triangle_cannot_hold():
    """A degenerate element (zero determinant: undefined entries) is stored
    whole, as the evaluation gives it."""
    pr = P.elastic_cube(1, nels_xyz=(11, 11, 10))
    gc = pr.g_coord().copy()
    gc[3] = 0.0
    with Context(0) as ctx:
        ctx.mesh_set(gc)
        ctx.steer_set(pr.g_g, pr.neq)
        ctx.assemble_elastic(pr.e, pr.v)
        K = ctx.storkm_get()
    assert np.isnan(K[3]).all()
    ok = [e for e in range(pr.nels) if e != 3]
    assert np.array_equal(K[ok], O.assemble_elastic(gc, pr.e, pr.v, nthreads=8)[ok])


def test_assembly_kept_whole_is_complete():
    """Moduli whose differences the triangle has no unit for: after the
    assembly into the triangle the matrices are formed whole, with their
    diagonal, and solved with as if they had been so at once."""
    pr = P.elastic_cube(1, nels_xyz=(11, 11, 10), lognormal_e=True)
    pr.e_elem = pr.e_elem.copy()
    pr.e_elem[17] = 1e-300
    print("[gpu-test] assembly kept whole", flush=True)
    with Context(0) as ctx:
        P.setup(ctx, pr)
        ctx.trim()
        assert ctx.mem_used() > pr.nels * 28800
        K = O.assemble_elastic(pr.g_coord(), pr.e, pr.v, pr.e_elem, nthreads=8)
        assert np.array_equal(ctx.storkm_get(), K)
        assert np.array_equal(ctx.diag_get(), O.diag(pr.g_g, K, pr.neq))
        assert np.array_equal(ctx.pcg_solve(pr.r0, 8, 0.0, stop="relres")[0], _oracle_iterates(pr, "relres", 8))


# p124's matrices on both sides of 32 MB (65,536 bricks), in wavefronts of a
# last workgroup that is partly filled, and with a material whose differences
# the triangle has no unit for (whole matrices then).
@pytest.mark.parametrize("box,tiny", [((32, 32, 64), False), ((65537, 1, 1), False), ((41, 40, 41), False),
                                      ((41, 40, 41), True)])
def test_transient_storage_bitexact(box, tiny):
    pr = _mesh_problem(8, box)
    rng = np.random.default_rng(11)
    pr.mesh.coords = pr.mesh.coords + rng.uniform(-0.15, 0.15, pr.mesh.coords.shape)
    gc = pr.mesh.g_coord()
    prop = np.array([[1.5, 0.7, 2.0, 1.2, 0.8], [0.4, 1.1, 0.3, 2.5, 1.7], [1e-290, 3e-290, 2e-290, 1e-160, 1e-140]])
    etype = rng.integers(1, 3, pr.nels).astype(np.int32)
    if tiny:
        etype[1000] = 3
    print(f"[gpu-test] transient storage {box} {tiny}", flush=True)
    KA, KB = O.assemble_transient(gc, prop, etype, 0.5, 0.01, nthreads=8)
    d = np.abs(KA[1000] - KA[1000].T).max()
    assert (0 < d < 2.0 ** -1008) == tiny       # a difference, and no unit below it
    x = rng.standard_normal(pr.neq)
    with Context(0) as ctx:
        ctx.mesh_set(gc)
        ctx.steer_set(pr.g_g, pr.neq)
        ctx.trim()
        before = ctx.mem_used()
        for _ in range(2):
            ctx.assemble_transient(0.5, 0.01, prop, etype)
        ctx.trim()
        # storkb whole; storka whole or as 372 bytes of 512
        held = ctx.mem_used() - before
        assert held >= 2 * KA.nbytes if tiny or pr.nels <= 65536 else held < 1.8 * KA.nbytes
        assert np.array_equal(ctx.storkm_get(), KA)
        dg = O.diag(pr.g_g, KA, pr.neq)
        assert np.array_equal(ctx.diag_get(), dg)
        assert np.array_equal(ctx.apply_raw(0, x), O.apply(pr.g_g, KA, x))
        assert np.array_equal(ctx.apply_raw(1, x), O.apply(pr.g_g, KB, x))
        xo = O.pcg(pr.g_g, KA, x, dg, 0.0, 5, stop=O.STOP_RELRES, dot_order=O.DOT_DEVICE, nthreads=8)[0]
        assert np.array_equal(ctx.pcg_solve(x, 5, 0.0, stop="relres")[0], xo)


@pytest.mark.parametrize("nod,box", [(20, (11, 11, 10)), (8, (20, 19, 20))])
def test_assembled_triangle_bitexact(nod, box):
    """Distorted elements with moduli of their own, assembled straight into
    the triangle: the oracle's matrices, diagonal and iterates."""
    if nod == 20:
        pr = P.elastic_cube(1, nels_xyz=box, lognormal_e=True)
    else:
        pr = _mesh_problem(24, box)
        pr.e_elem = M.lognormal(3, pr.nels, np.log(100.0), 0.5)
    rng = np.random.default_rng(2)
    pr.mesh.coords = pr.mesh.coords + rng.uniform(-0.15, 0.15, pr.mesh.coords.shape)
    print(f"[gpu-test] assembled triangle {nod} {box}", flush=True)
    with Context(0) as ctx:
        P.setup(ctx, pr)
        K = O.assemble_elastic(pr.g_coord(), pr.e, pr.v, pr.e_elem, nthreads=8)
        assert np.array_equal(ctx.storkm_get(), K)
        assert np.array_equal(ctx.diag_get(), O.diag(pr.g_g, K, pr.neq))
        for stop in ("checon", "relres"):
            x, _ = ctx.pcg_solve(pr.r0, 8, 0.0, stop=stop)
            assert np.array_equal(x, _oracle_iterates(pr, stop, 8))


# Node maps on both sides of the device's rule (65,536 slots and nodes), with a
# node of as many elements as the sort takes (64) and of one more, node numbers
# outside the mesh and a node without elements.
@pytest.mark.parametrize("nels", [2048, 7281, 7282, 20000])
@pytest.mark.parametrize("star", [0, 64, 65])
def test_node_maps(nels, star):
    rng = np.random.default_rng(nels + star)
    nod, nn = 8, 7287
    g = np.empty((nels, nod), dtype=np.int32)
    # every node but the last in at most 32 elements
    g[:] = np.resize(rng.permutation(nn - 1) + 1, (nels, nod))
    if star:
        g[g == 5] = 6
        g[rng.choice(nels, star, replace=False), 3] = 5
    g[1, 1], g[2, 2], g[3, 4] = 0, nn + 1, -3
    print(f"[gpu-test] node map nels={nels} star={star}", flush=True)
    with Context(0) as ctx:
        for numvar, flag in ((1, 1), (3, 0)):
            c = rng.standard_normal((nels, nod, numvar))
            assert np.array_equal(ctx.scatter_nodes(g, c, nn, flag), O.scatter_nodes(g, c, nn, flag), equal_nan=True)


# Lists that a thread sorts (16 slots) and that a workgroup does (17 to 4,096),
# more of them than workgroups, and one that is left to the host (4,097).
@pytest.mark.parametrize("length,count", [(16, 5), (17, 5), (255, 3), (256, 3), (257, 200), (4096, 2), (4097, 1)])
def test_node_maps_with_long_lists(length, count):
    rng = np.random.default_rng(length)
    nels, nod, nn = 20000, 8, 30000
    g = rng.permutation(np.resize(np.arange(1000, nn) + 1, nels * nod)).astype(np.int32)   # 5 or 6 each
    where = rng.choice(g.size, length * count, replace=False).reshape(count, length)
    for k in range(count):
        g[where[k]] = 1 + 3 * k
    g = g.reshape(nels, nod)
    print(f"[gpu-test] node lists {length} {count}", flush=True)
    with Context(0) as ctx:
        for numvar, flag in ((1, 1), (3, 0)):
            c = rng.standard_normal((nels, nod, numvar))
            assert np.array_equal(ctx.scatter_nodes(g, c, nn, flag), O.scatter_nodes(g, c, nn, flag), equal_nan=True)


# Elements of p122's stress update around the eight of a wavefront.
@pytest.mark.parametrize("nels", [1, 7, 8, 9, 67])
@pytest.mark.parametrize("phi", [0.0, 20.0])
def test_plastic_update_sizes(nels, phi):
    """Body loads, strains and stresses against the oracle to rounding
    (trigonometric functions: 1e-11 of each array's scale)."""
    m = M.box_hex8(nels, 1, 1, 0.5, 0.5, 0.5)
    rng = np.random.default_rng(nels)
    m.coords = m.coords + rng.uniform(-0.05, 0.05, m.coords.shape)
    nf, neq = M.steering(m.nn, 3, M.base_fixed_rest(m))
    g_g, gc = M.g_g_from(nf, m.g_num), m.g_coord()
    print(f"[gpu-test] plastic {nels} phi={phi}", flush=True)
    x = 1e-3 * rng.standard_normal(neq)
    evpt = 1e-5 * rng.standard_normal((nels, 8, 6))
    tensor = 20.0 * rng.standard_normal((nels, 8, 6))
    args = (1e4, 0.3, phi, 15.0, phi / 4, 5e-4)   # some points below yield
    with Context(0) as ctx:
        ctx.mesh_set(gc)
        ctx.steer_set(g_g, neq)
        dx, dev, dte = DeviceArray.from_host(ctx, x), DeviceArray.from_host(ctx, evpt), DeviceArray.from_host(ctx, tensor)
        dut = DeviceArray(ctx, nels * 24)
        for final in (False, True):
            ctx.plastic_update(dx, dev, dte, dut, *args, final)
            bl = O.plastic_update(gc, g_g, x, evpt, tensor, *args, final)
            got = dut.download().reshape(nels, 24)
            for a, b in ((got, bl), (dev.download().reshape(evpt.shape), evpt), (dte.download().reshape(tensor.shape), tensor)):
                assert np.abs(b).max() > 0 and np.abs(a - b).max() <= 1e-11 * np.abs(b).max(), final


# Solves whose replacements wait for the end of a run of six iterations, and
# the same iterations run one call at a time: p formed in the products or not
# (512 | 513 blocks), with fold launches (2,049 blocks) and with range-fused
# products (p formed in them and not), replacements between, on and right behind
# a run's end, limits that fall into a run, on its end and on a replacement.
@pytest.mark.parametrize("el,box,scatter", [(20, (4, 4, 4), "slots"), (24, (6, 5, 7), "slots"), (8, (31, 63, 63), "slots"),
                                            (8, (32, 63, 63), "slots"), (8, (64, 63, 127), "slots"),
                                            (20, (4, 4, 4), "ranges"), (8, (20, 15, 9), "ranges")])
@pytest.mark.parametrize("precision,every,delta,limit",
                         [("mixed", 0, 0.0, 20000), ("mixed64", 0, 0.1, 20000), ("mixed64", 0, 0.9, 40),
                          ("mixed", 6, 0.1, 60), ("mixed64", 7, 0.1, 61), ("mixed", 5, 0.1, 30), ("mixed64", 1, 0.5, 13)])
def test_parked_replacements(el, box, scatter, precision, every, delta, limit):
    if scatter == "ranges" and precision != "mixed":
        pytest.skip("range-fused products are the mixed solver's")
    if el == 20:
        pr = P.elastic_cube(1, nels_xyz=box, lognormal_e=True)
    elif el == 24:
        pr = _mesh_problem(24, box)
    else:
        pr = P.laplace_cube(1, nels_xyz=box)
    print(f"[gpu-test] parked {el} {box} {precision} {every} {delta} {limit}", flush=True)
    kw = dict(stop="relres", precision=precision, refine_delta=delta, refine_every=every)
    with Context(0) as ctx:
        r = P.setup(ctx, pr, store="fp32")
        ctx.scatter_mode = scatter
        x, res = ctx.pcg_solve(r, limit, 1e-9, **kw)
        ctx.pcg_begin(r, limit, 1e-9, **kw)
        while True:
            ctx.pcg_run(50)
            one = ctx.pcg_poll()
            if one.converged or one.iters >= limit:
                break
        assert (res.iters, res.refinements, res.converged) == (one.iters, one.refinements, one.converged)
        assert np.array_equal(x, ctx.pcg_x())
        # (limit 40 may end before the residual has fallen at all)
        assert res.refinements > 0 or limit == 40


# Replacements that nearly every iteration asks for keep their launches in every
# iteration (as many launches of them as of products); the others are launched
# once behind each run of iterations.
@pytest.mark.parametrize("delta,every,parks", [(0.0, 0, True), (0.5, 0, True), (0.5, 6, True), (0.51, 0, False),
                                               (0.9, 0, False), (0.1, 5, False)])
@pytest.mark.parametrize("box", [(12, 11, 10), (83, 81, 82)])       # without and with fold launches
def test_frequent_replacements_do_not_park(box, delta, every, parks):
    pr = P.laplace_cube(1, nels_xyz=box)
    print(f"[gpu-test] parks {box} {delta} {every}", flush=True)
    with Context(0) as ctx:
        r = P.setup(ctx, pr, store="fp32")
        ctx.timing_enable()
        res = ctx.pcg_solve(r, 60, 0.0, stop="relres", precision="mixed64", refine_delta=delta, refine_every=every)[1]
        t = ctx.timing_get()
        assert res.iters == 60
        assert (t["refine"][1] < t["ebe"][1]) == parks
        assert t["refine"][1] <= t["ebe"][1]


# Node freedom tables made on the device and on the host (the rule: 262,144
# element nodes and freedoms), with rows that a later one overrides.
@pytest.mark.parametrize("box", [(20, 20, 19), (28, 28, 29), (29, 28, 29), (60, 28, 30)])
@pytest.mark.parametrize("rows", ["none", "base", "twice"])
def test_node_freedoms(box, rows):
    m = M.box_hex8(*box)
    nod, n = 8, 3 * m.nn
    rng = np.random.default_rng(m.nn)
    rest = np.zeros((0, 4), dtype=np.int32)
    if rows != "none":
        rest = M.base_fixed_rest(m)
    if rows == "twice":     # some nodes again, in any order, with other freedoms
        again = rng.choice(m.nn, m.nn // 3, replace=True) + 1
        rest = np.concatenate([rest, np.column_stack([again, rng.integers(0, 2, (again.size, 3))])]).astype(np.int32)
    free = np.ones((m.nn, 3), dtype=bool)
    for row in rest:
        free[row[0] - 1] = row[1:] != 0
    nf = np.where(free.ravel(), np.cumsum(free.ravel()), 0).reshape(m.nn, 3)
    print(f"[gpu-test] node freedoms {box} {rows} {m.g_num.size + n}", flush=True)
    with Context(0) as ctx:
        ctx.mesh_set(m.g_coord())
        neq, got = ctx.steer_build(m.g_num, rest, m.nn)
        assert neq == nf.max() and np.array_equal(np.asarray(got).reshape(m.nn, 3), nf)
        assert np.array_equal(ctx.steer_get().reshape(m.nels, 24), M.g_g_from(nf, m.g_num).reshape(m.nels, 24))
        # what is refused leaves the steering as it is
        bad_num = m.g_num.copy()
        bad_num[-1, -1] = m.nn + 1
        bad_rest = np.concatenate([rest, np.array([[0, 1, 1, 1]], dtype=np.int32)]).astype(np.int32)
        every = np.column_stack([np.arange(1, m.nn + 1), np.zeros((m.nn, 3), dtype=int)]).astype(np.int32)
        for g, rs in ((bad_num, rest), (m.g_num, bad_rest), (m.g_num, every)):
            with pytest.raises(Exception):
                ctx.steer_build(g, rs, m.nn)
            assert np.array_equal(ctx.steer_get().reshape(m.nels, 24), M.g_g_from(nf, m.g_num).reshape(m.nels, 24))


# Slot lists of nodes (above 2,048 blocks of three-freedom nodes): freedoms
# restrained at random (leaders of each freedom, followers behind a gap), tied
# ones (lists that agree only in part), and a list too long for its code (the
# equations' own lists then).
@pytest.mark.parametrize("nf_kind", ["base", "random", "tied", "long"])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_node_slot_lists_bitexact(nf_kind, precision):
    pr = _mesh_problem(24, (2, 2, 20400))
    rng = np.random.default_rng(3)
    nf = pr.nf.copy()
    if nf_kind == "random":
        nf[rng.random(nf.shape) < 0.03] = 0
    elif nf_kind == "tied":         # z of every 50th node tied to z of the next
        a = np.arange(100, pr.mesh.nn - 1, 50)
        nf[a + 1, 2] = nf[a, 2]
    elif nf_kind == "long":         # one equation of 40 nodes
        a = np.arange(1000, 1040)
        nf[a, 0] = nf[1000, 0]
    nf = np.unique(nf, return_inverse=True)[1].reshape(nf.shape)   # 0 stays 0, equations consecutive
    neq = int(nf.max())
    assert (neq + 255) // 256 > 2048
    g_g = M.g_g_from(nf.astype(np.int32), pr.mesh.g_num)
    r = rng.standard_normal(neq)
    print(f"[gpu-test] node slot lists {nf_kind} {precision} neq={neq}", flush=True)
    with Context(0) as ctx:
        ctx.mesh_set(pr.mesh.g_coord())
        ctx.steer_set(g_g, neq)
        ctx.assemble_elastic(100.0, 0.3, store="fp64" if precision == "fp64" else "fp32")
        x, res = ctx.pcg_solve(r, 4, 0.0, stop="relres", precision=precision)
        K = O.assemble_elastic(pr.mesh.g_coord(), 100.0, 0.3, nthreads=8)
        xo = O.pcg(g_g, K, r, O.diag(g_g, K, neq), 0.0, 4, stop=O.STOP_RELRES, dot_order=O.DOT_DEVICE)[0]
        if precision == "fp64":
            assert np.array_equal(x, xo)
        else:
            # FP32 products: 24 terms of 8 elements at 2^-24, four iterations
            assert np.abs(x - xo).max() <= 4 * 24 * 8 * 2.0 ** -24 * np.abs(xo).max()


# What the server admits a request by, on both sides of the padded slot table
# (2,048 blocks: 34 | 35) and of whole FP64 matrices (32 MB: 10 | 11).
@pytest.mark.parametrize("n", [1, 10, 11, 34, 35, 50])
@pytest.mark.parametrize("precision", ["mixed64", "fp64"])
def test_admission_counts_what_a_request_holds(n, precision):
    from parafem_amd import serve as S
    d = S.CubeCache().get(n)
    print(f"[gpu-test] device bytes {n} {precision}", flush=True)
    with Context(0) as ctx:
        ctx.mesh_set(d["g_coord"])
        ctx.steer_build(d["g_num"], d["rest"], d["nn"])
        ctx.assemble_elastic(100.0, 0.3, store="fp64" if precision == "fp64" else "fp32")
        ctx.pcg_begin(d["r_unit"], 10, 0.0, stop="relres", precision=precision)
        assert ctx.mem_used() <= S.device_bytes(n, precision)
        ctx.pcg_run(2)
        assert ctx.pcg_poll().iters == 2


# The product that an iteration runs, on both sides of the storage's and the
# iteration's rules, and the bytes it reads an element.
@pytest.mark.parametrize("ntot,box,store,precision,stop,want", [
    (60, (3, 1, 2), "fp64", "fp64", "checon", ("k_ebe_form<60, 0, double, 1>", 1, False, 28800 + 240)),
    (60, (12, 12, 12), "fp64", "fp64", "relres", ("k_ebe<60, 5, true, double, false, 1>", 1, False, 18364 + 240)),
    (60, (12, 12, 12), "fp32", "mixed", "relres", ("k_ebe_form<60, 1, float, 2>", 1, False, 7328 + 240)),
    (60, (24, 24, 24), "fp32", "mixed", "relres", ("k_ebe<60, 1, true, float, false, 1>", 1, True, 7328 + 240)),
    (60, (24, 24, 24), "fp32", "split", "checon", ("k_ebe<60, 2, true, double, false, 1>", 1, True, 14656 + 240)),
    (24, (20, 19, 20), "fp64", "fp64", "relres", ("k_ebe<24, 5, true, double, false, 1>", 1, False, 2496 + 532 + 96)),
    (8, (20, 20, 20), "fp64", "fp64", "relres", ("k_ebe_form<8, 4, double, 2>", 2, False, 320 + 32)),
    (8, (60, 60, 60), "fp64", "fp64", "relres", ("k_ebe<8, 4, true, double, false, 2>", 2, False, 320 + 32)),
    (8, (60, 60, 60), "fp32", "mixed64", "relres", ("k_ebe<8, 3, true, double, false, 4>", 4, True, 144 + 32))])
def test_product_that_an_iteration_runs(ntot, box, store, precision, stop, want):
    pr = _mesh_problem(ntot, box)
    print(f"[gpu-test] product {ntot} {box} {precision}", flush=True)
    with Context(0) as ctx:
        P.setup(ctx, pr, store=store)
        got = ctx.ebe_kernel(precision, stop)
        assert (got["kernel"], got["epl"], got["tunable"], got["bytes_per_element"]) == want
        if got["tunable"]:
            ctx.tune_set(ebe_epl=2)
            assert ctx.ebe_kernel(precision, stop)["epl"] == 2
        with pytest.raises(Exception):
            ctx.ebe_kernel("fp64" if store == "fp32" else "mixed", stop)
