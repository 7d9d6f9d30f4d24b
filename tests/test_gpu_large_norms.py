"""Residual norms where their route changes with the tree's size: one tree's
partials summed in pieces (above 32,768), 3D levels without sibling groups beside
grouped ones (above 3,000 leaves in a launch of their own), levels whose leaves are
some of their blocks, and column levels of more than 80,000 blocks. Against the
oracle to 1e-12 (its sum in another order), and the norm that a mixed solve forms
with its defects against the norm alone."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")  # noqa: F841  (torch's HIP runtime first)

from oracle import Oracle
from srmg import configs, solver
from srmg.solver import F32, F64

pytestmark = pytest.mark.gpu

BCS = {2: ((1, -1), (-1, 1)), 3: ((1, -1), (-1, -1), (-1, 1))}
corner = lambda l, c: np.all(c <= 2, axis=1)  # noqa: E731


@pytest.mark.parametrize("D,root,M,levels,geom", [
    (2, (256, 128), 8, 1, 1), (2, (256, 129), 8, 1, 0), (2, (257, 130), 8, 2, 2), (2, (31, 33), 16, 2, 1),
    (3, (15, 15, 13), 8, 2, 0), (3, (15, 15, 15), 8, 2, 0), (3, (14, 14, 14), 8, 1, 0), (3, (5, 4, 3), 16, 2, 0)])
def test_norm_follows_the_oracle(D, root, M, levels, geom):
    print(f"norm D={D} root={root} M={M} levels={levels}", flush=True)
    p = configs.uniform_problem(D, root, M, levels, geom, BCS[D], refine=corner, G=1)
    g, disc = solver.geometry_from_code(p.geom), solver.LaplacianDiscretization(D, 2)
    ctx = solver.Context(p.tree, p.conn, p.M)
    u, b, r, _ = (ctx.field(F64) for _ in range(4))
    o = Oracle.for_problem(p)
    uo = p.b.like()
    uo.u[...] = np.random.default_rng(6).normal(size=uo.u.shape)
    o.fill_ghost_all(uo)
    u.upload(uo)
    b.upload(p.b)
    n = solver.resnorm(r, b, u, p.s, geometry=g, bc=p.bc, lpldisc=disc)
    assert n == pytest.approx(o.resnorm(p.b.like(), p.b.copy(), uo, p.s), rel=1e-12)
    v, w = ctx.field(F32), ctx.field(F32)
    v.upload(uo)
    w.upload(p.b)
    # FP32: residuals of order one from terms of order one to ten, an RMS over many cells
    assert solver.resnorm(r, w, v, p.s, geometry=g, bc=p.bc, lpldisc=disc) == pytest.approx(n, rel=1e-5)


@pytest.mark.parametrize("root,refine", [((15, 15, 15), corner), ((22, 22, 22), lambda l, c: c[:, 0] >= 1)])
def test_norm_with_the_defects_is_the_norm(root, refine):
    p = configs.uniform_problem(3, root, 8, 2, 0, BCS[3], refine=refine, G=1)
    print(f"defects root={root}: {[len(x) for x in p.tree]} blocks", flush=True)
    g, disc = solver.geometry_from_code(p.geom), solver.LaplacianDiscretization(3, 2)
    ctx = solver.Context(p.tree, p.conn, p.M)
    u, b, r = (ctx.field(F64) for _ in range(3))
    e = [ctx.field(F32) for _ in range(4)]
    b.upload(p.b)
    n0 = solver.resnorm(r, b, u, p.s, geometry=g, bc=p.bc, lpldisc=disc)
    n, h = solver.solve_mixed(u, b, *e, p.s, g, p.bc, disc, tol=0.0, max_cycles=3, coarse=solver.COARSE_GS)
    # covered cells of b hold the right-hand sides of the FAS cycles: the norm is of the leaves
    n1 = solver.resnorm(r, b, u, p.s, geometry=g, bc=p.bc, lpldisc=disc)
    assert h[0] == pytest.approx(1.0, rel=1e-12)
    assert n1 == pytest.approx(h[-1] * n0, rel=1e-12)
