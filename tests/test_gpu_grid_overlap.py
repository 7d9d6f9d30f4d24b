"""Level-1 grids solved into a buffer that lies across the right-hand sides'
(shifted by planes, by part of a row, by whole grids): the same bits as into a
buffer of its own. Many stacked grids, which are otherwise solved in place, and
few; with and without device allocations."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from srmg import configs, solver
from srmg.tree import boundaryconditions

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,grids", [((16, 8, 64), 8), ((8, 8, 8), 64), ((16, 16, 16), 4)])
@pytest.mark.parametrize("shift", [3, 64, -128, 1024, -4096])
@pytest.mark.parametrize("noalloc", [False, True])
def test_result_across_the_right_hand_side(n, grids, shift, noalloc):
    print(f"grids {n} x {grids}, shift {shift}, noalloc {noalloc}", flush=True)
    p = configs.uniform_problem(2, (1, 2), 16, 1, 0, ((1, 1), (-1, -1)))
    ctx = solver.Context(p.tree, p.conn, p.M)
    bc = boundaryconditions(((1, -1), (1, 1), (-1, -1)))
    geom, disc = solver.CartesianGeometry(), solver.LaplacianDiscretization(3, 2)
    total = int(np.prod(n)) * grids
    rhs = torch.tensor(np.random.default_rng(4).normal(size=total), device="cuda")
    own = torch.empty_like(rhs)
    solver.grid_solve(ctx, 3, n, 1.0, geom, bc, disc, rhs, own, grids)
    both = torch.zeros(total + abs(shift), dtype=torch.float64, device="cuda")
    f, u = both[max(0, -shift):][:total], both[max(0, shift):][:total]
    f.copy_(rhs)
    torch.cuda.synchronize()
    solver.grid_solve(ctx, 3, n, 1.0, geom, bc, disc, f, u, grids, noalloc=noalloc)
    torch.cuda.synchronize()
    assert torch.isfinite(own).all() and torch.equal(u, own)
