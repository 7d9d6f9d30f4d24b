"""Coarse-fine ghost slabs of all levels in one launch, or level by level where
a slab is interpolated from another one (a refined block without a diagonal
neighbour): ghost fills and the cycles that follow against the oracle, bit for
bit."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")  # noqa: F841  (torch's HIP runtime first)

from oracle import Oracle
from srmg import configs, solver
from srmg.solver import F64

pytestmark = pytest.mark.gpu


def _tree(D, M, diagonal):
    roots = [(2, 2), (1, 2), (2, 1)] + ([(1, 1)] if diagonal else [])

    def crit(l, c):
        if l == 1:
            return np.array([tuple(q[:2]) in roots for q in c.tolist()])
        return np.all(c[:, :2] == 3, axis=1) & (l == 2)
    return configs.uniform_problem(D, (4,) * D, M, 3, 0, ((1, -1),) * D, refine=crit)


@pytest.mark.parametrize("D,M", [(2, 16), (2, 8), (3, 8)])
@pytest.mark.parametrize("diagonal", [True, False])
def test_filled_slabs_follow_the_oracle(D, M, diagonal):
    p = _tree(D, M, diagonal)
    assert len(p.tree) == 3 and len(p.tree[2].pairs) > 0
    geom, disc = solver.geometry_from_code(p.geom), solver.LaplacianDiscretization(D, 2)
    ctx = solver.Context(p.tree, p.conn, p.M)
    u, b, r, u1 = (ctx.field(F64) for _ in range(4))
    o = Oracle.for_problem(p)
    uo, bo, ro, u1o = p.b.like(), p.b.copy(), p.b.like(), p.b.like()
    vs = (slice(p.b.G, p.b.G + M),) * D
    uo.u[vs] = np.random.default_rng(3).standard_normal(uo.u[vs].shape)
    b.upload(p.b)
    u.upload(uo)
    got = p.b.like()
    for _ in range(2):
        solver.fill_ghost_all(u, p.bc)
        o.fill_ghost_all(uo)
        assert solver.resnorm(r, b, u, p.s, geometry=geom, bc=p.bc, lpldisc=disc) == pytest.approx(
            o.resnorm(p.b.like(), bo, uo, p.s), rel=1e-12)
        solver.vcycle(u, b, r, u1, p.s, geometry=geom, bc=p.bc, lpldisc=disc, ndown=2, ntop=4, nup=2)
        o.vcycle(uo, bo, ro, u1o, p.s, ndown=2, ntop=4, nup=2)
        u.download(got)
        np.testing.assert_array_equal(got.u[vs], uo.u[vs])
