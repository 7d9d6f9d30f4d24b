"""Single V-cycles replayed as a graph from their third call on: each replay
against the oracle, bit for bit, with eager work on the same fields in between
(uploads, fills, norms, sweeps that leave a field in its second buffer), other
configurations and more of them than are kept, and a forest."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")  # noqa: F841  (torch's HIP runtime first)

from oracle import Oracle
from srmg import configs, solver
from srmg.solver import F64
from srmg.tree import box_stencil, connectivity

pytestmark = pytest.mark.gpu


def _vs(p):
    return (slice(p.b.G, p.b.G + p.M),) * p.D


@pytest.mark.parametrize("coarse", [solver.COARSE_GS, solver.COARSE_EXACT])
def test_replayed_cycles_follow_the_oracle(coarse):
    p = configs.make_cfg1(2)
    geom, disc = solver.geometry_from_code(p.geom), solver.LaplacianDiscretization(2, 2)
    ctx = solver.Context(p.tree, p.conn, p.M)
    u, b, r, u1, w = (ctx.field(F64) for _ in range(5))
    b.upload(p.b)
    o = Oracle.for_problem(p)
    uo, bo, ro, u1o = p.b.like(), p.b.copy(), p.b.like(), p.b.like()
    other = solver.HelmholtzDiscretization(2, 2, 3.0e5)
    for it in range(9):
        nup = 3 if it % 4 == 3 else 2  # another configuration now and then
        solver.fill_ghost_all(u, p.bc)
        solver.vcycle(u, b, r, u1, p.s, geometry=geom, bc=p.bc, lpldisc=disc, ndown=2, ntop=4, nup=nup, coarse=coarse)
        o.fill_ghost_all(uo)
        o.vcycle(uo, bo, ro, u1o, p.s, ndown=2, ntop=4, nup=nup, coarse_exact=coarse == solver.COARSE_EXACT)
        n = solver.resnorm(r, b, u, p.s, geometry=geom, bc=p.bc, lpldisc=disc)
        assert n == pytest.approx(o.resnorm(p.b.like(), bo, uo, p.s), rel=1e-12)
        got = u.download(p.b.like())
        np.testing.assert_array_equal(got.u[_vs(p)], uo.u[_vs(p)])
        if it == 4:  # another problem's matrices and parameters in between
            v, c = ctx.field(F64), ctx.field(F64).upload(p.b)
            solver.vcycle(v, c, r, u1, p.s, geometry=geom, bc=np.ones(9, np.int8), lpldisc=other, coarse=coarse)
            v.close()  # drops what was captured
        if it == 6:
            u.upload(got)  # the ghosts of coarse-fine faces come with it
            for k in range(70):  # more configurations than are kept
                solver.vcycle(w, b, r, u1, p.s, geometry=geom, bc=p.bc, lpldisc=disc, ndown=0, ntop=0,
                              nup=0, omega=1.0 + k / 100, coarse=solver.COARSE_GS)
            b.upload(p.b)
            bo.u[...] = p.b.u


def test_replayed_forest_cycles_equal_single_trees():
    probs = configs.make_helmholtz_cfg1(1)
    geom = solver.geometry_from_code(probs[0].geom)
    discs = [solver.HelmholtzDiscretization(2, 2, p.k2) for p in probs]
    ctx = solver.Context.forest([(p.tree, p.conn) for p in probs], probs[0].M)
    u, b, r, u1 = (ctx.field(F64) for _ in range(4))
    b.upload(solver.concat_fields([p.b for p in probs]))
    orc = [(Oracle.for_problem(p), p.b.like(), p.b.copy(), p.b.like(), p.b.like()) for p in probs]
    G, M = probs[0].b.G, probs[0].M
    for it in range(5):
        solver.vcycle_batched(u, b, r, u1, [p.s for p in probs], geom, probs[0].bc, discs, ndown=2, ntop=4, nup=2)
        got = np.zeros((M,) * 2 + (ctx.nblocks,), order="F")
        u.download(got)
        for p, (o, uo, bo, ro, u1o), v in zip(probs, orc, solver.split_field(got, [p.tree.nblocks() for p in probs])):
            o.vcycle(uo, bo, ro, u1o, p.s, ndown=2, ntop=4, nup=2)
            np.testing.assert_array_equal(v, uo.u[G:G + M, G:G + M])


def test_replayed_order4_cycles_follow_the_oracle():
    p = configs.uniform_problem(2, (4, 4), 16, 3, 0, ((1, -1), (-1, -1)))
    geom, disc = solver.geometry_from_code(p.geom), solver.LaplacianDiscretization(2, 4)
    ctx = solver.Context(p.tree, p.conn, p.M)
    u, q, q1, r, u1 = (ctx.field(F64) for _ in range(5))
    q.upload(p.b)
    solver.rhs(q1, q, geom, p.bc, disc)
    o = Oracle(p.tree, connectivity(p.tree, box_stencil(2)), p.M, p.b.G, p.geom, p.bc, order=4)
    uo, qo, q1o, ro, u1o = p.b.like(), p.b.copy(), p.b.like(), p.b.like(), p.b.like()
    o.rhs(q1o, qo, order=4)
    got = p.b.like()
    for _ in range(6):
        solver.fill_ghost_all(u, p.bc, disc)
        solver.vcycle(u, q1, r, u1, p.s, p.tree, p.conn, geom, p.bc, disc, ndown=1, ntop=3, nup=2)
        o.fill_ghost_all(uo)
        o.vcycle(uo, q1o, ro, u1o, p.s, ndown=1, ntop=3, nup=2)
        u.download(got)
        np.testing.assert_array_equal(got.u[_vs(p)], uo.u[_vs(p)])
