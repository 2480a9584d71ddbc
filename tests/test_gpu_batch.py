"""Batched iterations (pf_batch_*): several solves of different sizes
advanced by one launch per kernel.  Bars: every solve's iteration count and
displacements bit-identical to the same solve run alone on its context
(pf_pcg_solve), in every precision, with checon and residual stopping; the
FP64 solves also bit-identical to the oracle in the device's reduction order
(p121.f90:89-104 / p123.f90:135-151 per solve)."""
import sys

import numpy as np
import pytest

import oracle as O
from parafem_amd import Batch, Context, problems as P

pytestmark = pytest.mark.gpu


def say(msg):
    print(f"[gpu-test] {msg}", flush=True)
    sys.stdout.flush()


def _elastic_mix():
    out = []
    for n, e, v, q in ((3, 100.0, 0.3, 1.0), (5, 37.0, 0.22, 4.0), (2, 150.0, 0.35, 0.3), (4, 80.0, 0.28, 2.5)):
        out.append(P.elastic_cube(n, e=e, v=v, pressure=q))
    out.append(P.elastic_cube(4, lognormal_e=True))
    return out


def _run_batch(ctxs, rs, limit, tol, stop, precision, graph, chunk=7, solo=0):
    """graph: True (replayed graph), False (direct launches) or
    "persistent" (one cooperative kernel per chunk); solo: solves of at
    least that many elements run their own launches in the batch."""
    for c, r in zip(ctxs, rs):
        c.pcg_begin(r, limit, tol, stop=stop, precision=precision)
    b = Batch(0)
    try:
        b.solo_set(solo)
        live = list(range(len(ctxs)))
        done = {}
        while live:
            b.run([ctxs[k] for k in live], chunk, graph=graph is True, persistent=graph == "persistent")
            got = None
            while got is None:
                got = b.query()
            snap, res = got
            assert [c.h for c in snap] == [ctxs[k].h for k in live]
            keep = []
            for k, rr in zip(live, res):
                if rr.converged or rr.status == 6 or rr.iters >= limit:
                    done[k] = (rr.iters, bool(rr.converged), ctxs[k].pcg_x())
                else:
                    keep.append(k)
            live = keep       # the set shrinks as solves finish
        return [done[k] for k in range(len(ctxs))]
    finally:
        b.close()


@pytest.mark.parametrize("precision,stop,graph", [("fp64", "checon", True), ("fp64", "relres", False),
                                                  ("split", "relres", True), ("mixed64", "relres", True),
                                                  ("mixed", "relres", True), ("mixed", "relres", False),
                                                  ("fp64", "checon", "persistent"),
                                                  ("split", "relres", "persistent"),
                                                  ("mixed64", "relres", "persistent"),
                                                  ("mixed", "relres", "persistent")])
def test_batch_equals_alone_hex20(precision, stop, graph):
    probs = _elastic_mix()
    store = "fp64" if precision == "fp64" else "fp32"
    tol = 1e-7 if stop == "checon" else 1e-10
    ctxs = [Context(0) for _ in probs]
    try:
        rs = [P.setup(c, pr, store=store) for c, pr in zip(ctxs, probs)]
        say(f"batch hex20 {precision} {stop} graph={graph}: alone")
        alone = []
        for c, r in zip(ctxs, rs):
            x, res = c.pcg_solve(r, 3000, tol, stop=stop, precision=precision)
            alone.append((res.iters, res.converged, x))
        say(f"batch hex20 {precision} {stop} graph={graph}: batched")
        got = _run_batch(ctxs, rs, 3000, tol, stop, precision, graph)
        for (ia, ca, xa), (ib, cb, xb) in zip(alone, got):
            assert ca and cb and ia == ib
            assert np.array_equal(xa, xb)
        if precision == "fp64":
            pr = probs[1]
            Ko = O.assemble_elastic(pr.g_coord(), pr.e, pr.v, pr.e_elem)
            so = O.STOP_CHECON if stop == "checon" else O.STOP_RELRES
            xo, it, conv = O.pcg(pr.g_g, Ko, pr.r0, O.diag(pr.g_g, Ko, pr.neq), tol, 3000, stop=so,
                                 dot_order=O.DOT_DEVICE)
            assert it == got[1][0] and np.array_equal(xo, got[1][2])
    finally:
        for c in ctxs:
            c.close()


@pytest.mark.parametrize("precision,graph", [("fp64", True), ("mixed", True), ("fp64", "persistent"),
                                             ("mixed", "persistent")])
def test_batch_equals_alone_hex8_laplace_penalty(precision, graph):
    """hex8 Laplace cubes with penalty fixed freedoms (p123's fixed rows in
    the scatter) and, for the mixed path, the FP32 copy of p."""
    probs = [P.laplace_cube(n, lognormal_k=True, seed=s) for n, s in ((5, 2), (3, 7), (7, 9))]
    store = "fp64" if precision == "fp64" else "fp32"
    ctxs = [Context(0) for _ in probs]
    try:
        rs = [P.setup(c, pr, store=store) for c, pr in zip(ctxs, probs)]
        say(f"batch hex8 laplace {precision}: alone")
        alone = [c.pcg_solve(r, 3000, 1e-10, stop="relres", precision=precision) for c, r in zip(ctxs, rs)]
        say(f"batch hex8 laplace {precision} {graph}: batched")
        got = _run_batch(ctxs, rs, 3000, 1e-10, "relres", precision, graph, chunk=5)
        for (xa, ra), (ib, cb, xb) in zip(alone, got):
            assert ra.converged and cb and ra.iters == ib
            assert np.array_equal(xa, xb)
    finally:
        for c in ctxs:
            c.close()


@pytest.mark.parametrize("precision,stop,graph,solo", [("mixed64", "relres", True, 60), ("fp64", "checon", False, 60),
                                                       ("mixed", "relres", True, 1), ("split", "relres", True, 100)])
def test_batch_with_solo_solves_equals_alone(precision, stop, graph, solo):
    """Solves above the solo threshold run their own launches inside the
    batch's runs (all of them for threshold 1), the rest share the batched
    launches: every solve still bit-identical to itself alone."""
    probs = _elastic_mix()
    store = "fp64" if precision == "fp64" else "fp32"
    tol = 1e-7 if stop == "checon" else 1e-10
    ctxs = [Context(0) for _ in probs]
    try:
        rs = [P.setup(c, pr, store=store) for c, pr in zip(ctxs, probs)]
        say(f"batch solo>={solo} {precision} {stop} graph={graph}: alone")
        alone = []
        for c, r in zip(ctxs, rs):
            x, res = c.pcg_solve(r, 3000, tol, stop=stop, precision=precision)
            alone.append((res.iters, res.converged, x))
        say(f"batch solo>={solo} {precision} {stop} graph={graph}: batched")
        got = _run_batch(ctxs, rs, 3000, tol, stop, precision, graph, solo=solo)
        for (ia, ca, xa), (ib, cb, xb) in zip(alone, got):
            assert ca and cb and ia == ib
            assert np.array_equal(xa, xb)
    finally:
        for c in ctxs:
            c.close()


@pytest.mark.parametrize("el,precision,stop", [("hex20", "fp64", "checon"), ("hex20", "mixed64", "relres"),
                                               ("hex8", "fp64", "relres"), ("hex8", "mixed", "relres"),
                                               ("hex8", "split", "checon")])
def test_persistent_with_more_blocks_than_workgroups(el, precision, stop):
    """Solves of more equation blocks (256 equations) than workgroups are
    resident (at most 8 a CU, 2,048), so that a workgroup sums one block after
    another: the iterates of every solve alone, bit for bit."""
    if el == "hex20":
        probs = [P.elastic_cube(n) for n in (31, 8, 30, 5)]
    else:
        probs = [P.laplace_cube(n, lognormal_k=True, seed=n) for n in (70, 12, 66, 5)]
    assert sum((pr.neq + 255) // 256 for pr in probs) > 2048
    store = "fp64" if precision == "fp64" else "fp32"
    ctxs = [Context(0) for _ in probs]
    try:
        rs = [P.setup(c, pr, store=store) for c, pr in zip(ctxs, probs)]
        say(f"persistent {el} {precision} {stop}: alone")
        kw = dict(stop=stop, precision=precision)
        if precision.startswith("mixed"):
            kw["refine_delta"] = 0.5          # some replacements among the 24 iterations
        alone = [c.pcg_solve(r, 24, 0.0, **kw) for c, r in zip(ctxs, rs)]
        for c, r in zip(ctxs, rs):
            c.pcg_begin(r, 24, 0.0, **kw)
        say(f"persistent {el} {precision} {stop}: batched")
        with Batch(0) as b:
            for _ in range(3):
                b.run(ctxs, 9, persistent=True)
            for c, (x, res) in zip(ctxs, alone):
                got = c.pcg_poll()
                assert (got.iters, got.refinements) == (res.iters, res.refinements) and res.iters == 24
                assert np.array_equal(c.pcg_x(), x)
    finally:
        for c in ctxs:
            c.close()


@pytest.mark.parametrize("precision,n", [("mixed64", 18), ("mixed", 18), ("mixed64", 34), ("mixed", 34)])
def test_batch_replacements(precision, n):
    """Solves of very different sizes whose residuals are replaced in the same
    and in different iterations, more blocks of products than workgroups; below
    1 GiB of matrices (dealt to the solves) and above (every workgroup on each
    solve in turn): every solve as alone, replacements counted alike."""
    probs = [P.elastic_cube(n, e=37.0, v=0.22), P.elastic_cube(2), P.elastic_cube(9, lognormal_e=True),
             P.elastic_cube(n, e=74.0, v=0.22), P.elastic_cube(5, v=0.4)]
    assert (sum(pr.nels for pr in probs) * 14656 > 1 << 30) == (n == 34) and (probs[0].neq + 255) // 256 <= 2048
    ctxs = [Context(0) for _ in probs]
    try:
        rs = [P.setup(c, pr, store="fp32") for c, pr in zip(ctxs, probs)]
        say(f"batch replacements {precision} {n}")
        # (the residuals of the large solves have not fallen yet: every 40 iterations)
        kw = dict(stop="relres", precision=precision, refine_delta=0.5, refine_every=40)
        alone = [c.pcg_solve(r, 90, 0.0, **kw) for c, r in zip(ctxs, rs)]
        assert min(res.refinements for _, res in alone) > 0
        with Batch(0) as b:
            for graph in (True, False):
                for c, r in zip(ctxs, rs):
                    c.pcg_begin(r, 90, 0.0, **kw)
                for _ in range(6):
                    b.run(ctxs, 16, graph=graph)
                for c, (x, res) in zip(ctxs, alone):
                    got = c.pcg_poll()
                    assert (got.iters, got.refinements) == (res.iters, res.refinements)
                    assert np.array_equal(c.pcg_x(), x)
    finally:
        for c in ctxs:
            c.close()


@pytest.mark.parametrize("precision,stop", [("fp64", "checon"), ("mixed64", "relres"), ("mixed", "relres")])
def test_batch_of_solves_with_and_without_folds(precision, stop):
    """A solve above 2,048 reduction blocks joins and leaves a batch of solves
    below (which then fold by launches, or for themselves): the iterates of
    every solve alone, whichever way each run took."""
    probs = [P.laplace_cube(n, lognormal_k=True, seed=n) for n in (12, 81, 30, 5)]
    assert (probs[1].neq + 255) // 256 > 2048 >= (probs[2].neq + 255) // 256
    ctxs = [Context(0) for _ in probs]
    try:
        rs = [P.setup(c, pr, store="fp64" if precision == "fp64" else "fp32") for c, pr in zip(ctxs, probs)]
        say(f"batch with and without folds {precision}")
        kw = dict(stop=stop, precision=precision)
        if precision != "fp64":
            kw["refine_delta"] = 0.5
        alone = [c.pcg_solve(r, 30, 0.0, **kw) for c, r in zip(ctxs, rs)]
        small = [ctxs[0], ctxs[2], ctxs[3]]
        with Batch(0) as b:
            for graph in (True, False):
                for c, r in zip(ctxs, rs):
                    c.pcg_begin(r, 30, 0.0, **kw)
                b.run(small, 7, graph=graph)
                b.run(ctxs, 11, graph=graph)
                b.run(small, 5, graph=graph)
                b.run(ctxs, 30, graph=graph)
                for c, (x, res) in zip(ctxs, alone):
                    got = c.pcg_poll()
                    assert (got.iters, got.refinements) == (res.iters, res.refinements) and res.iters == 30
                    assert np.array_equal(c.pcg_x(), x)
    finally:
        for c in ctxs:
            c.close()


def test_batch_rejects_mixed_settings():
    """Solves of one batch share ntot, precision and stopping rule."""
    from parafem_amd import PFError
    a, b = Context(0), Context(0)
    try:
        ra = P.setup(a, P.elastic_cube(2))
        rb = P.setup(b, P.elastic_cube(3))
        a.pcg_begin(ra, 100, 1e-8, stop="relres")
        b.pcg_begin(rb, 100, 1e-8, stop="checon")
        with Batch(0) as bt:
            with pytest.raises(PFError):
                bt.run([a, b], 2)
            with pytest.raises(PFError):
                bt.run([a, a], 2)
    finally:
        a.close()
        b.close()
