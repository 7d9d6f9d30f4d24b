"""Two sweeps in one launch (2D) against the oracle, bit for bit: random trees
(concave corners of refined levels, boundaries on every side), both block sizes
and geometries, odd and even numbers of sweeps, and the FP32 path against two
launches of one sweep each."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")  # noqa: F841  (torch's HIP runtime first)

from oracle import Oracle
from srmg import configs, solver
from srmg.solver import F32, F64
from regrid_cases import problem

pytestmark = pytest.mark.gpu


def _trees():
    out = {f"random{s}": (lambda s=s: configs.make_random_tree_problem(s)) for s in (0, 1, 2, 3, 4, 5)}
    out["amr"] = lambda: problem(2)
    out["one-block"] = lambda: configs.uniform_problem(2, (1, 1), 8, 1, 1, ((1, -1), (-1, 1)))
    out["strip"] = lambda: configs.uniform_problem(2, (1, 5), 16, 1, 2, ((-1, 1), (1, 1)))
    return out


TREES = _trees()


@pytest.mark.parametrize("name", list(TREES))
@pytest.mark.parametrize("sweeps", [(2, 4, 2), (3, 5, 3), (1, 2, 5)])
def test_pairs_follow_the_oracle(name, sweeps):
    p = TREES[name]()
    ndown, ntop, nup = sweeps
    geom, disc = solver.geometry_from_code(p.geom), solver.LaplacianDiscretization(2, 2)
    ctx = solver.Context(p.tree, p.conn, p.M)
    u, b, r, u1 = (ctx.field(F64) for _ in range(4))
    b.upload(p.b)
    o = Oracle.for_problem(p)
    uo, bo, ro, u1o = p.b.like(), p.b.copy(), p.b.like(), p.b.like()
    vs = (slice(p.b.G, p.b.G + p.M),) * 2
    got = p.b.like()
    for _ in range(2):
        solver.fill_ghost_all(u, p.bc)
        solver.vcycle(u, b, r, u1, p.s, geometry=geom, bc=p.bc, lpldisc=disc, ndown=ndown, ntop=ntop, nup=nup)
        o.fill_ghost_all(uo)
        o.vcycle(uo, bo, ro, u1o, p.s, ndown=ndown, ntop=ntop, nup=nup)
        u.download(got)
        np.testing.assert_array_equal(got.u[vs], uo.u[vs])


@pytest.mark.parametrize("name", list(TREES))
def test_pairs_equal_single_sweeps(name):
    p = TREES[name]()
    geom, disc = solver.geometry_from_code(p.geom), solver.LaplacianDiscretization(2, 2)
    ctx = solver.Context(p.tree, p.conn, p.M)
    res = []
    for steps in ((4,), (1, 1, 1, 1)):
        u, b, r, u1 = (ctx.field(F32) for _ in range(4))
        b.upload(p.b)
        u.upload(p.b)
        solver.fill_ghost_all(u, p.bc)
        for n in steps:  # the coarsest level alone
            solver.vcycle(u, b, r, u1, p.s, geometry=geom, bc=p.bc, lpldisc=disc, lmax=1, ndown=0, ntop=n, nup=0)
        got = p.b.like()
        u.download(got)
        res.append(got.u.copy())
        for f in (u, b, r, u1):
            f.close()
    np.testing.assert_array_equal(res[0], res[1])
