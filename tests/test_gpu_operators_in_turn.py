"""Two operators in turn on one context, as a time step has them (the potential,
then photoionization with another boundary table): V-cycles with the exact
level-1 solve, whose matrices the context holds for one boundary table at a
time, called often enough that each would be replayed, against the oracle, bit
for bit; and solves whose first step is replayed after another operator's."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")  # noqa: F841  (torch's HIP runtime first)

from oracle import Oracle
from srmg import configs, solver
from srmg.solver import F64
from srmg.tree import boundaryconditions

pytestmark = pytest.mark.gpu

OTHER = {2: ((1, 1), (-1, -1)), 3: ((-1, -1), (-1, -1), (-1, -1))}  # the second operator's boundaries


def _problem(D):
    if D == 2:
        return configs.make_cfg1(2)
    crit = lambda l, c: np.all(c <= 2 ** (l - 1), axis=1)  # noqa: E731
    return configs.uniform_problem(3, (2, 2, 2), 8, 3, 0, ((1, -1), (-1, -1), (1, 1)), refine=crit)


class _Run:
    """One operator's fields on the shared context, and the oracle's."""

    def __init__(self, p, ctx, bc, k2=None):
        self.p, self.bc = p, bc
        self.geom = solver.geometry_from_code(p.geom)
        self.disc = solver.LaplacianDiscretization(p.D, 2) if k2 is None else solver.HelmholtzDiscretization(p.D, 2, k2)
        self.f = [ctx.field(F64) for _ in range(4)]
        self.f[1].upload(p.b)
        self.o = Oracle(p.tree, p.conn, p.M, p.b.G, p.geom, bc, k2 is not None, k2 or 0.0)
        self.fo = [p.b.like(), p.b.copy(), p.b.like(), p.b.like()]
        self.vs = (slice(p.b.G, p.b.G + p.M),) * p.D

    def cycle(self):
        solver.fill_ghost_all(self.f[0], self.bc)
        solver.vcycle(*self.f, self.p.s, geometry=self.geom, bc=self.bc, lpldisc=self.disc, ndown=2, ntop=4, nup=2,
                      coarse=solver.COARSE_EXACT)
        self.o.fill_ghost_all(self.fo[0])
        self.o.vcycle(*self.fo, self.p.s, ndown=2, ntop=4, nup=2, coarse_exact=True)
        got = self.f[0].download(self.p.b.like())
        np.testing.assert_array_equal(got.u[self.vs], self.fo[0].u[self.vs])

    def solve(self, **kw):
        return solver.solve(*self.f, self.p.s, self.geom, self.bc, self.disc, tol=1e-8, max_cycles=4, **kw)


@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("order", ["AABA", "ABABABABABAB", "AABBAABBAABB", "AAAABAAAABBBBA"])
def test_vcycles_of_two_boundary_tables(D, order):
    p = _problem(D)
    ctx = solver.Context(p.tree, p.conn, p.M)
    runs = {"A": _Run(p, ctx, p.bc), "B": _Run(p, ctx, boundaryconditions(OTHER[D]), 3.0e4)}
    for k in order:
        runs[k].cycle()


@pytest.mark.parametrize("per_step", [1, 2, 3])
def test_vcycles_between_solves_of_another_boundary_table(per_step):
    p = _problem(2)
    ctx = solver.Context(p.tree, p.conn, p.M)
    a, b = _Run(p, ctx, p.bc), _Run(p, ctx, boundaryconditions(OTHER[2]), 3.0e4)
    ref = None
    for _ in range(4):
        for _ in range(per_step):
            a.cycle()
        b.f[0].zero()
        n, hist = b.solve()
        ref = hist if ref is None else ref
        np.testing.assert_array_equal(hist, ref)


def test_first_fmg_step_replayed_after_another_operator():
    p = _problem(2)
    ctx = solver.Context(p.tree, p.conn, p.M)
    a, b = _Run(p, ctx, p.bc), _Run(p, ctx, boundaryconditions(OTHER[2]), 3.0e4)

    def solve(r, **kw):
        r.f[1].upload(p.b)
        r.f[0].zero()
        n, hist = r.solve(first_fmg=True, **kw)
        return hist, r.f[0].download(p.b.like()).u[r.vs].copy()

    h0, u0 = solve(a, use_graph=False)
    for _ in range(3):
        solve(b)
        h, u = solve(a, use_graph=True)
        np.testing.assert_array_equal(h, h0)
        np.testing.assert_array_equal(u, u0)
