"""2D levels one sweep to a launch (odd numbers of sweeps; even ones go in pairs
whatever tile shape is set): every tile shape against the oracle in FP64 and
against each other in FP32, on trees and forests with sibling groups, both radial
dimensions; and pairs against single sweeps on refined levels, where they read
coarse-fine slabs, across faces of either direction and around concave corners of
the level, in both precisions. All bit for bit."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")  # noqa: F841  (torch's HIP runtime first)

from oracle import Oracle
from srmg import configs, solver
from srmg.solver import F32, F64
from test_gpu_parity import CASES, _disc

pytestmark = pytest.mark.gpu

ODD = dict(ndown=1, ntop=3, nup=1)
SHAPED = {k: CASES[k] for k in ("cfg1", "cyl1-m16", "cyl2-m8", "cart2-helm")}
# complete sibling groups on every refined level, radial dimension 2
SHAPED["cyl2-m16-groups"] = lambda: configs.uniform_problem(2, (2, 4), 16, 3, 2, ((1, -1), (1, -1)),
                                                            refine=lambda l, c: c[:, 1] <= 2)


def _vs(p):
    return (slice(p.b.G, p.b.G + p.M),) * p.D


@pytest.mark.parametrize("name", list(SHAPED))
@pytest.mark.parametrize("dtype", [F64, F32])
def test_every_shape_of_a_single_sweep(name, dtype):
    p = SHAPED[name]()
    print(f"single sweeps {name} dtype {dtype}", flush=True)
    geom, disc = solver.geometry_from_code(p.geom), _disc(p)
    outs = []
    for cfg in range(solver.SWEEP_SHAPES):
        ctx = solver.Context(p.tree, p.conn, p.M)
        u, b, r, u1 = (ctx.field(dtype) for _ in range(4))
        for l in range(1, len(p.tree) + 1):
            ctx.set_sweep_config(dtype, l, cfg)
        b.upload(p.b)
        solver.fill_ghost_all(u, p.bc)
        for _ in range(2):
            solver.vcycle(u, b, r, u1, p.s, geometry=geom, bc=p.bc, lpldisc=disc, **ODD)
        outs.append(u.download(p.b.like()).u[_vs(p)].copy())
        ctx.close()
    for o in outs[1:]:
        np.testing.assert_array_equal(o, outs[0])
    if dtype == F64:
        o = Oracle.for_problem(p)
        uo, bo, ro, u1o = p.b.like(), p.b.copy(), p.b.like(), p.b.like()
        o.fill_ghost_all(uo)
        for _ in range(2):
            o.vcycle(uo, bo, ro, u1o, p.s, **ODD)
        np.testing.assert_array_equal(outs[0], uo.u[_vs(p)])


@pytest.mark.parametrize("cfg", [0, 1, 2, 3, 4, 5, 6])
def test_single_sweeps_of_a_forest(cfg):
    probs = configs.make_helmholtz_cfg1(1) + configs.make_helmholtz_cfg1(2)[:1]
    geom = solver.geometry_from_code(probs[0].geom)
    discs = [_disc(p) for p in probs]
    ctx = solver.Context.forest([(p.tree, p.conn) for p in probs], probs[0].M)
    u, b, r, u1 = (ctx.field(F64) for _ in range(4))
    for l in range(1, max(len(p.tree) for p in probs) + 1):
        ctx.set_sweep_config(F64, l, cfg)
    b.upload(solver.concat_fields([p.b for p in probs]))
    solver.fill_ghost_all(u, probs[0].bc)
    for _ in range(2):
        solver.vcycle_batched(u, b, r, u1, [p.s for p in probs], geom, probs[0].bc, discs, **ODD)
    G, M = probs[0].b.G, probs[0].M
    got = np.zeros((M,) * 2 + (ctx.nblocks,), order="F")
    u.download(got)
    for p, v in zip(probs, solver.split_field(got, [p.tree.nblocks() for p in probs])):
        o, uo, bo, ro, u1o = Oracle.for_problem(p), p.b.like(), p.b.copy(), p.b.like(), p.b.like()
        o.fill_ghost_all(uo)
        for _ in range(2):
            o.vcycle(uo, bo, ro, u1o, p.s, **ODD)
        np.testing.assert_array_equal(v, uo.u[G:G + M, G:G + M])


@pytest.mark.parametrize("M", [8, 16])
@pytest.mark.parametrize("geom", [0, 1, 2])
@pytest.mark.parametrize("seed", [0, 1, 2])
@pytest.mark.parametrize("dtype", [F64, F32])
def test_pairs_equal_single_sweeps_on_a_refined_level(M, geom, seed, dtype):
    rng = np.random.default_rng(seed)
    root = (5, 6) if seed else (7, 3)
    marks = rng.uniform(size=root) < (0.45, 0.6, 0.75)[seed]
    p = configs.uniform_problem(2, root, M, 2, geom, ((1, -1), (-1, 1)),
                                refine=lambda l, c: marks[c[:, 0] - 1, c[:, 1] - 1])
    print(f"pairs M={M} geom={geom} seed={seed}: {[len(x) for x in p.tree]} blocks", flush=True)
    g, disc = solver.geometry_from_code(p.geom), solver.LaplacianDiscretization(2, 2)
    ctx = solver.Context(p.tree, p.conn, p.M)
    start = p.b.like()
    start.u[...] = rng.normal(size=start.u.shape)
    fine = np.array([b for _, b in p.tree[1].pairs]) - 1
    outs = []
    for pairs in (True, False):
        u, b, r, u1 = (ctx.field(dtype) for _ in range(4))
        b.upload(p.b)
        u.upload(start)
        solver.fill_ghost_all(u, p.bc)
        if pairs:
            # without sweeps on level 1 the correction is zero: level 2 keeps its eight sweeps
            solver.vcycle(u, b, r, u1, p.s, geometry=g, bc=p.bc, lpldisc=disc, ndown=8, ntop=0, nup=0)
        else:
            # two launches, then two captured ones replayed three times
            ctx.time_kernel(solver.KERNEL_GS_SWEEP, 2, u, b, r, p.s, g, p.bc, disc, reps=2)
        outs.append(u.download(p.b.like()).u[_vs(p) + (fine,)].copy())
        for f in (u, b, r, u1):
            f.close()
    assert np.isfinite(outs[0]).all() and np.abs(outs[0] - start.u[_vs(p) + (fine,)]).max() > 0
    np.testing.assert_array_equal(outs[0], outs[1])
