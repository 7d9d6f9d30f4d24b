"""The one-launch four-colour sweeps of 2D levels against the oracle, bit for
bit: odd numbers of sweeps (the values end in the second buffer), cycles on a
new iterate without a ghost fill before them (the first pass reads the ghosts
as they were), one level alone, and the trees' coarse-fine corners."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")  # noqa: F841  (torch's HIP runtime first)

from test_gpu_order4 import AMR, CASES, GEOM
from oracle import Oracle
from srmg import solver
from srmg.solver import F64
from srmg.tree import box_stencil, connectivity

pytestmark = pytest.mark.gpu

TREES = {**{k: (lambda f=f, k=k: (f(), GEOM[k])) for k, f in CASES.items() if not k.startswith("3d")},
         **{k: f for k, f in AMR.items() if f()[0].D == 2}}


@pytest.mark.parametrize("name", list(TREES))
@pytest.mark.parametrize("sweeps", [(1, 3, 2), (2, 1, 3), (0, 2, 1)])
def test_sweeps_without_a_fill_follow_the_oracle(name, sweeps):
    p, gcode = TREES[name]()
    ndown, ntop, nup = sweeps
    geom, disc = solver.geometry_from_code(gcode), solver.LaplacianDiscretization(2, 4)
    ctx = solver.Context(p.tree, p.conn, p.M)
    u, b, r, u1 = (ctx.field(F64) for _ in range(4))
    b.upload(p.b)
    o = Oracle(p.tree, connectivity(p.tree, box_stencil(2)), p.M, p.b.G, gcode, p.bc, order=4)
    uo, bo, ro, u1o = p.b.like(), p.b.copy(), p.b.like(), p.b.like()
    vs = (slice(p.b.G, p.b.G + p.M),) * 2
    rng = np.random.default_rng(5)
    got = p.b.like()
    for it, lmax in enumerate((0, 0, 1, 0)):
        if it % 2:  # a new iterate, its ghosts as the last cycle left them
            uo.u[vs] = rng.standard_normal(uo.u[vs].shape)
            got.u[...] = uo.u
            u.upload(got)
        solver.vcycle(u, b, r, u1, p.s, p.tree, p.conn, geom, p.bc, disc, lmax=lmax, ndown=ndown, ntop=ntop, nup=nup)
        o.vcycle(uo, bo, ro, u1o, p.s, lmax=lmax, ndown=ndown, ntop=ntop, nup=nup)
        u.download(got)
        np.testing.assert_array_equal(got.u[vs], uo.u[vs])
