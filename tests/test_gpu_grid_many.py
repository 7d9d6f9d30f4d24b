"""Stacked level-1 grids: whole planes per work group (512 z planes and more)
against the axis-by-axis kernels, bit for bit, at the smallest and largest
extents, extents whose rows do not share out evenly over the waves, with the
Helmholtz shift and in place."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from srmg import configs, solver
from srmg.tree import boundaryconditions

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,grids", [((8, 8, 8), 64), ((64, 64, 64), 8), ((64, 32, 32), 16), ((24, 40, 56), 10),
                                     ((56, 8, 16), 33)])
def test_many_grids_equal_the_axis_kernels(n, grids):
    print(f"grids {n} x {grids}", flush=True)
    p = configs.uniform_problem(2, (1, 2), 16, 1, 0, ((1, 1), (-1, -1)))
    ctx = solver.Context(p.tree, p.conn, p.M)
    bc = boundaryconditions(((1, -1), (1, 1), (-1, -1)))
    geom, disc = solver.CartesianGeometry(), solver.HelmholtzDiscretization(3, 2, 2.0e4)
    f = torch.tensor(np.random.default_rng(2).normal(size=(grids, int(np.prod(n)))), device="cuda")
    many, axes = torch.full_like(f, float("nan")), torch.full_like(f, float("nan"))
    solver.grid_solve(ctx, 3, n, 1e-6, geom, bc, disc, f, many, grids)
    ctx.set_axis_gemm(1)
    solver.grid_solve(ctx, 3, n, 1e-6, geom, bc, disc, f, axes, grids)
    ctx.set_axis_gemm(2)
    torch.cuda.synchronize()
    assert torch.isfinite(axes).all() and torch.equal(many, axes)
    solver.grid_solve(ctx, 3, n, 1e-6, geom, bc, disc, f, f, grids)
    torch.cuda.synchronize()
    assert torch.equal(f, axes)
