"""Trees of many levels (more than one launch of the all-level norms takes, and
an odd number) against the oracle: V-cycles bit for bit, the norm to 1e-12 (its
sums in another fixed order), with level 1 of one shape or several, grouped or
not, both coarse treatments, FP64 and the mixed solve (1e-7, as documented)."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")  # noqa: F841  (torch's HIP runtime first)

from oracle import Oracle
from srmg import configs, solver
from srmg.solver import F32, F64

pytestmark = pytest.mark.gpu

# D, root, M, levels, geometry, boundary
CASES = [(2, (1, 2), 16, 15, 1, ((1, -1), (-1, -1))), (2, (2, 2), 16, 13, 0, ((1, -1), (-1, 1))),
         (2, (3, 2), 8, 14, 2, ((-1, -1), (1, -1))), (3, (1, 2, 1), 8, 7, 0, ((1, 1), (-1, 1), (-1, -1)))]


def _problem(D, root, M, levels, geom, bc):
    return configs.uniform_problem(D, root, M, levels, geom, bc, refine=lambda l, c: np.all(c == 1, axis=1))


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}d-m{c[2]}-{c[3]}")
@pytest.mark.parametrize("coarse", [solver.COARSE_GS, solver.COARSE_EXACT])
def test_deep_tree_cycles_and_norms(case, coarse):
    p = _problem(*case)
    print(f"deep tree {case}: {p.tree.nblocks()} blocks", flush=True)
    geom, disc = solver.geometry_from_code(p.geom), solver.LaplacianDiscretization(p.D, 2)
    ctx = solver.Context(p.tree, p.conn, p.M)
    u, b, r, u1 = (ctx.field(F64) for _ in range(4))
    b.upload(p.b)
    o = Oracle.for_problem(p)
    uo, bo, ro, u1o = p.b.like(), p.b.copy(), p.b.like(), p.b.like()
    G, M = p.b.G, p.M
    vs = (slice(G, G + M),) * p.D
    for it in range(3):
        solver.fill_ghost_all(u, p.bc)
        solver.vcycle(u, b, r, u1, p.s, geometry=geom, bc=p.bc, lpldisc=disc, ndown=2, ntop=4, nup=2 + it % 2,
                      coarse=coarse)
        o.fill_ghost_all(uo)
        o.vcycle(uo, bo, ro, u1o, p.s, ndown=2, ntop=4, nup=2 + it % 2, coarse_exact=coarse == solver.COARSE_EXACT)
        got, gb = p.b.like(), p.b.like()
        u.download(got)
        b.download(gb)
        np.testing.assert_array_equal(got.u[vs], uo.u[vs])
        np.testing.assert_array_equal(gb.u[vs], bo.u[vs])
        n = solver.resnorm(r, b, u, p.s, geometry=geom, bc=p.bc, lpldisc=disc)
        assert n == pytest.approx(o.resnorm(p.b.like(), bo, uo, p.s), rel=1e-12)


@pytest.mark.parametrize("case", CASES[:2] + CASES[3:], ids=lambda c: f"{c[0]}d-m{c[2]}-{c[3]}")
def test_deep_tree_mixed_solve(case):
    p = _problem(*case)
    geom, disc = solver.geometry_from_code(p.geom), solver.LaplacianDiscretization(p.D, 2)
    ctx = solver.Context(p.tree, p.conn, p.M)
    u, b, r, u1 = (ctx.field(F64) for _ in range(4))
    e, be, re, ue = (ctx.field(F32) for _ in range(4))
    vs = (slice(p.b.G, p.b.G + p.M),) * p.D
    out = []
    for mixed in (False, True):
        b.upload(p.b)
        if mixed:
            solver.solve_mixed(u, b, e, be, re, ue, p.s, geom, p.bc, disc, tol=1e-10, max_cycles=40,
                               guess=solver.GUESS_ZERO)
        else:
            solver.solve(u, b, r, u1, p.s, geom, p.bc, disc, tol=1e-10, max_cycles=40, guess=solver.GUESS_ZERO)
        out.append(u.download(p.b.like()).u[vs].copy())
    assert np.max(np.abs(out[1] - out[0])) <= 1e-7 * np.max(np.abs(out[0]))
