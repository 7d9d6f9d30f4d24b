"""Performance cases of the elliptic solvers, through their public entry points.

What a streamer code and the learned first iterate's recipe have the library do:

poisson   the Poisson block of a time step: the charge q restricted, the
          right-hand side formed, a few warm-started V-cycles with the
          reference's level-1 sweeps; order 2 or the compact order 4
solve     a Poisson solve to 1e-8 of the initial residual, FP64 or FP32 with
          FP64 defect correction
photo     the photoionization Helmholtz terms (on one tree, optionally with
          other trees in the same launches), solved to 1e-8
dropin    one V-cycle on host arrays, as a caller that keeps the reference's
          host fields replaces vcycle!: upload, cycle, download
grid      exact level-1 solves of stacked uniform grids (training targets)
infer     the network's prediction
train     one training step of the network

Fields live on the device between calls, as a resident caller keeps them: a
pass hands them back as device-resident outputs that are copied to the host
when they are looked at (:class:`Resident`).

``exact`` is the same arithmetic in 64 bits written with torch tensors: the
V-cycle, the converged solve, the level-1 solve, the network.
"""

import functools
import math
import os

import numpy as np
import torch

from __graft_entry__ import ROOT, load_package

load_package()
from srmg import configs, solver  # noqa: E402
from srmg.tree import boundaryconditions, connectivity, refined_tree  # noqa: E402

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64, F32 = solver.F64, solver.F32
TOL = 1e-8
NETS = {"cfg2": (2, (128, 256, 1)), "cfg4": (3, (64, 64, 64))}


def listed():
    return [
        # the axisymmetric Gaussian cloud: 4 x 8 root blocks of 16^2, three
        # levels, about 20k cells; the reference's poisson_iter = 2
        dict(name="poisson-small", kind="poisson", D=2, M=16, geom=1, r0=4, r1=8, r2=1, levels=3, blocks=76, iters=2,
             order=2),
        # the same block with the compact fourth-order operator
        dict(name="poisson-order4", kind="poisson", D=2, M=16, geom=1, r0=4, r1=8, r2=1, levels=3, blocks=76,
             iters=2, order=4),
        # the axisymmetric streamer tree: 8 x 16 root blocks, six levels, 2M cells
        dict(name="solve2d-fp64", kind="solve", D=2, M=16, geom=1, r0=8, r1=16, r2=1, levels=6, blocks=7736,
             form="fp64"),
        dict(name="solve2d-mixed", kind="solve", D=2, M=16, geom=1, r0=8, r1=16, r2=1, levels=6, blocks=7736,
             form="mixed"),
        # a 3D tree with an odd, uneven root, four levels, 4M cells
        dict(name="solve3d-fp64", kind="solve", D=3, M=8, geom=0, r0=5, r1=6, r2=7, levels=4, blocks=8000,
             form="fp64"),
        # the benchmark's size: 8^3 root blocks of 8^3, five levels, 32M cells
        dict(name="solve3d-large", kind="solve", D=3, M=8, geom=0, r0=8, r1=8, r2=8, levels=5, blocks=62000,
             form="mixed"),
        # photoionization!: its three terms on the small tree
        dict(name="photo-terms", kind="photo", r0=4, r1=8, levels=3, blocks=76, trees=0, form="fp64"),
        # the terms together with 24 independent trees of many sizes
        dict(name="photo-forest", kind="photo", r0=4, r1=8, levels=3, blocks=76, trees=24, form="mixed"),
        # the drop-in vcycle! on the host fields of the streamer tree
        dict(name="dropin", kind="dropin", D=2, M=16, geom=1, r0=8, r1=16, r2=1, levels=6, blocks=7736),
        # one chunk of training targets of the 3D network
        dict(name="grid-targets", kind="grid", D=3, geom=0, n0=64, n1=64, n2=64, grids=128),
        # the first iterate of a 3D solve
        dict(name="net-infer", kind="infer", net="cfg4", batch=1),
        # the 3D training recipe's batch
        dict(name="net-train", kind="train", net="cfg4", batch=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["poisson", "poisson", "solve", "solve", "solve", "photo", "dropin", "grid", "infer", "train"])
    if kind == "grid":
        if rng.random() < 0.5:
            n = [rng.choice([24, 32, 40, 48, 64, 50]) for _ in range(3)]
            return dict(kind=kind, D=3, geom=0, n0=n[0], n1=n[1], n2=n[2], grids=_log(rng, 1, 128))
        return dict(kind=kind, D=2, geom=rng.choice([0, 1, 2]), n0=rng.randint(16, 128), n1=rng.randint(16, 256), n2=1,
                    grids=_log(rng, 1, 512))
    if kind == "infer":
        return dict(kind=kind, net=rng.choice(["cfg2", "cfg4"]), batch=_log(rng, 1, 24))
    if kind == "train":
        return dict(kind=kind, net=rng.choice(["cfg2", "cfg4"]), batch=_log(rng, 1, 16))
    if kind == "photo":
        r0 = rng.randint(2, 6)
        lv = rng.randint(2, 5)
        return dict(kind=kind, r0=r0, r1=rng.randint(r0, 2 * r0), levels=lv, blocks=_log(rng, 60, 2000),
                    trees=rng.choice([0, 0, rng.randint(1, 24)]), form=rng.choice(["fp64", "mixed"]))
    D = 2 if kind == "dropin" else rng.choice([2, 3])
    if D == 2:
        r0 = rng.randint(2, 8)
        c = dict(kind=kind, D=2, M=rng.choice([8, 16, 16]), geom=rng.choice([0, 1, 1, 2]), r0=r0,
                 r1=rng.randint(r0, 2 * r0), r2=1, levels=rng.randint(2, 6), blocks=_log(rng, 40, 7700))
    else:
        c = dict(kind=kind, D=3, M=8, geom=0, r0=rng.randint(3, 8), r1=rng.randint(3, 8), r2=rng.randint(3, 8),
                 levels=rng.randint(2, 4), blocks=_log(rng, 300, 12000))
    if kind == "poisson":
        c.update(iters=rng.randint(1, 3), order=rng.choice([2, 2, 4]))
    if kind == "solve":
        c.update(form=rng.choice(["fp64", "mixed"]))
    return c


# ---- trees and charges ----

def _spine(D, seed):
    """The curve that a tree is refined around, in units of the domain: the
    axis of the first dimension in 2D, slanted filaments in 3D."""
    r = np.random.default_rng(seed)
    if D == 2:
        z0, z1 = r.uniform(0.25, 0.45), r.uniform(0.6, 0.75)
        return [(np.array([0.0, z0]), np.array([0.0, z1]))]
    return [(np.array([r.uniform(0.3, 0.7), r.uniform(0.3, 0.7), 0.85]),
             np.array([r.uniform(0.3, 0.7), r.uniform(0.3, 0.7), 0.2])) for _ in range(3)]


@functools.lru_cache(maxsize=64)
def _tree(D, M, root, levels, blocks, seed=0):
    """A tree of about `blocks` blocks: at every level the blocks nearest to
    the spine are refined, in equal proportion; the neighbours of a refined
    block (diagonal ones too, as the order-4 operator needs) exist."""
    n1 = int(np.prod(root))
    lo, hi = 0.0, float(2 ** D)
    for _ in range(60):  # blocks per level grow by this factor
        g = 0.5 * (lo + hi)
        lo, hi = (g, hi) if n1 * sum(g ** k for k in range(levels)) < blocks else (lo, g)
    frac = min(0.95, g / 2 ** D)
    spine = _spine(D, seed)
    refined = []
    have = np.stack(np.meshgrid(*[np.arange(n) for n in root], indexing="ij"), -1).reshape(-1, D)
    step = np.stack(np.meshgrid(*[[0, 1]] * D, indexing="ij"), -1).reshape(-1, D)
    around = np.stack(np.meshgrid(*[[-1, 0, 1]] * D, indexing="ij"), -1).reshape(-1, D)
    for l in range(levels - 1):
        c = (have + 0.5) / (np.array(root) << l)
        d = np.full(len(c), np.inf)
        for a, b in spine:
            t = np.clip(((c - a) @ (b - a)) / ((b - a) @ (b - a)), 0, 1)
            d = np.minimum(d, np.linalg.norm(c - a - t[:, None] * (b - a), axis=1))
        take = have[np.argsort(d, kind="stable")[:max(1, int(round(frac * len(have))))]]
        refined.append(take)
        have = (2 * take[:, None, :] + step).reshape(-1, D)
    for l in range(levels - 2, 0, -1):  # properly nested, finest level first
        q = (refined[l][:, None, :] + around).reshape(-1, D)
        q = np.vstack([q, refined[l]])
        q = q[np.all((q >= 0) & (q < (np.array(root) << l)), axis=1)] >> 1
        refined[l - 1] = np.unique(np.vstack([refined[l - 1], q]), axis=0)
    sets = [set(map(tuple, (r + 1).tolist())) for r in refined]
    tree = refined_tree(D, root, levels, lambda lvl, cs: np.array([tuple(x) in sets[lvl - 1] for x in cs.tolist()]))
    return tree, connectivity(tree)


def _root(case):
    return tuple(case[k] for k in ("r0", "r1", "r2")[:case["D"]])


def _setup(case, t=0):
    """(tree, conn, operator pieces) of tree t of the case."""
    if case["kind"] == "photo":
        if t < 3:
            D, M, root, levels, blocks, seed = 2, 16, (case["r0"], case["r1"]), case["levels"], case["blocks"], 0
        else:  # uneven companions: 1e4 to 1e6 cells, two to six levels
            r = np.random.default_rng(100 + t)
            rx = int(r.integers(1, 5))
            D, M, root, levels, seed = 2, 16, (rx, 2 * rx), int(r.integers(2, 7)), t
            blocks = int(max(2 * rx * rx + 8, 10 ** r.uniform(1.6, 3.6)))
        geom, bc = 1, boundaryconditions(((1, 1), (-1, -1)))
        k2 = float(configs.bourdon3_terms()[1][t % 3])
    else:
        D, M, root, levels, blocks, seed = case["D"], case["M"], _root(case), case["levels"], case["blocks"], 0
        geom, k2 = case["geom"], None
        if D == 3:
            bc = boundaryconditions(((1, 1), (1, 1), (-1, -1)))
        else:  # Neumann on the axis, Dirichlet elsewhere
            bc = boundaryconditions(((-1, -1), (1, -1)) if geom == 2 else ((1, -1), (-1, -1)))
    tree, conn = _tree(D, M, root, levels, blocks, seed)
    h = (5e-3 if D == 2 else 1e-2) / (root[0] * M)
    s = h * h if k2 is not None else h * h * configs.ELEMENTARY_CHARGE / configs.EPSILON_0
    return dict(tree=tree, conn=conn, D=D, M=M, root=root, geom=geom, bc=np.asarray(bc, np.int8).ravel(), k2=k2, h=h,
                s=s, spine=_spine(D, seed))


def _ntrees(case):
    return 3 + case["trees"] if case["kind"] == "photo" else 1


def _charge(p, seed):
    """[blocks, (z,) y, x] FP64 on DEV: Gaussian clouds along the spine,
    evaluated at the cell centres of every block of every level."""
    D, M, r = p["D"], p["M"], np.random.default_rng(seed)
    nblk = p["tree"].nblocks()
    clouds = []
    for _ in range(12):
        a, b = p["spine"][r.integers(len(p["spine"]))]
        clouds.append((10 ** r.uniform(18, 20), a + r.uniform(0, 1) * (b - a), r.uniform(0.02, 0.06)))
    out = torch.empty((nblk,) + (M,) * D, dtype=torch.float64, device=DEV)
    off = (torch.arange(M, device=DEV, dtype=torch.float64) + 0.5) / M
    for l, layer in enumerate(p["tree"]):
        if not len(layer):
            continue
        co = torch.tensor([c for c, _ in layer.pairs], device=DEV, dtype=torch.float64)
        bl = torch.tensor([b for _, b in layer.pairs], device=DEV) - 1
        acc = 0.0
        for amp, c, w in clouds:
            v = amp
            for d in range(D):
                # lengths in units of the first dimension's
                x = (co[:, d:d + 1] - 1 + off) / (p["root"][0] << l) - c[d] * p["root"][d] / p["root"][0]
                shape = [len(bl)] + [M if e == D - 1 - d else 1 for e in range(D)]
                v = v * torch.exp(-(x / w) ** 2).reshape(shape)
            acc = acc + v
        out[bl] = acc
    return out


def _host(a, D, G):
    """[blocks, (z,) y, x] to the reference's host layout with G ghost layers."""
    a = torch.nn.functional.pad(a, (G, G) * D)
    return a.cpu().numpy().transpose(tuple(range(D, -1, -1)))


class Resident(dict):
    """Outputs of a pass that stay on the device: read from there when asked for."""

    def __getitem__(self, k):
        v = dict.__getitem__(self, k)
        return v() if callable(v) else v


def _read(f):
    """The valid cells of a device field, in the host layout without ghosts."""
    c = f.ctx
    return f.download(np.empty((c.M,) * c.D + (c.nblocks,), np.float64, order="F"))


# ---- the level-1 grids and the network's inputs ----

def _grid_charges(n, geom, count, seed, width):
    """[count, V] FP64, x fastest: Gaussian clouds and, on half of them, the axis."""
    r = np.random.default_rng(seed)
    D = len(n)
    out = torch.empty((count,) + tuple(reversed(n)), dtype=torch.float64, device=DEV)
    ax = [(torch.arange(m, device=DEV, dtype=torch.float64) + 0.5) / m for m in n]
    for k in range(count):
        acc = 0.0
        for _ in range(int(r.integers(1, 13))):
            v = 10 ** r.uniform(18, 21) * (-1 if r.uniform() < 0.3 else 1)
            for d in range(D):
                c = r.uniform(0.0, 0.05) if geom == d + 1 and r.uniform() < 0.5 else r.uniform(0.1, 0.9)
                e = torch.exp(-((ax[d] - c) / (width * r.uniform(0.5, 2.0))) ** 2)
                v = v * e.reshape([n[d] if D - 1 - d == a else 1 for a in range(D)])
            acc = acc + v
        out[k] = acc
    return out.reshape(count, -1)


def _grid_bc(D, geom):
    if D == 3:
        return ((1, 1), (1, 1), (-1, -1))
    return ((-1, -1), (1, -1)) if geom == 2 else ((1, -1), (-1, -1))


def _axis(n, radial, lo, hi):
    """The 1D operator of one axis as P diag(lam) Q (mirror ghosts folded in)."""
    i = torch.arange(1, n + 1, dtype=torch.float64)
    w = 2 * i - 1 if radial else torch.ones(n, dtype=torch.float64)
    up = 2 * i if radial else torch.ones(n, dtype=torch.float64)
    dg = torch.full((n,), -2.0, dtype=torch.float64)
    dg[0] += 0.0 if radial else lo
    dg[-1] += (up / w)[-1] * hi
    off = up[:-1] / torch.sqrt(w[:-1] * w[1:])
    lam, Y = torch.linalg.eigh(torch.diag(dg) + torch.diag(off, 1) + torch.diag(off, -1))
    return lam.to(DEV), (Y / torch.sqrt(w)[:, None]).to(DEV), (Y.T * torch.sqrt(w)).to(DEV)


def _level1(f, n, geom, bcd, shift=0.0):
    """L_1 u = f on stacked grids f [count, (z,) y, x]."""
    D = len(n)
    A = [_axis(n[d], geom == d + 1, *map(float, bcd[d])) for d in range(D)]
    lam = 0.0
    for d in range(D):
        f = torch.movedim(torch.movedim(f, D - d, -1) @ A[d][2].T, -1, D - d)
        lam = lam + A[d][0].reshape([n[d] if D - 1 - d == a else 1 for a in range(D)])
    f = f / (lam + shift)
    for d in range(D):
        f = torch.movedim(torch.movedim(f, D - d, -1) @ A[d][1].T, -1, D - d)
    return f


def _net_inputs(case, seed):
    """(f, u) FP32 [batch, V]: level-1 problems and their solutions."""
    D, n = NETS[case["net"]]
    n, geom = n[:D], 1 if D == 2 else 0
    h = 1e-2 / n[0]
    b = _grid_charges(n, geom, case["batch"], seed, 0.05)
    f = -h * h * configs.ELEMENTARY_CHARGE / configs.EPSILON_0 * b
    shape = (case["batch"],) + tuple(reversed(n))
    u = _level1(f.reshape(shape), n, geom, _grid_bc(D, geom)).reshape(f.shape)
    return f.float().contiguous(), u.float().contiguous()


def _weights(case):
    with np.load(os.path.join(ROOT, "steamroller.jl_amd", "weights", f"unet_{case['net']}_level1.npz")) as z:
        return z["params"].copy(), float(z["output_scale"]), tuple(int(x) for x in z["widths"])


# ---- the cases ----

def prepare(case, seed):
    kind = case["kind"]
    if kind == "grid":
        D = case["D"]
        n = [case["n0"], case["n1"], case["n2"]][:D]
        tree, conn = _tree(2, 16, (1, 2), 1, 2)
        st = dict(case=case, ctx=solver.Context(tree, conn, 16), n=n, geom=solver.geometry_from_code(case["geom"]),
                  bc=boundaryconditions(_grid_bc(D, case["geom"])), disc=solver.LaplacianDiscretization(D, 2),
                  s=(1e-2 / n[0]) ** 2 * configs.ELEMENTARY_CHARGE / configs.EPSILON_0)
        st["f"] = -st["s"] * _grid_charges(n, case["geom"], case["grids"], seed, 0.05)
        st["u"] = torch.empty_like(st["f"])
        return st
    if kind in ("infer", "train"):
        par, scale, widths = _weights(case)
        D, n = NETS[case["net"]]
        net = solver.UNet(D, n[:D], len(widths), widths)
        net.set_params(par if kind == "infer" else _first_weights(case, seed))
        net.output_scale = scale
        f, u = _net_inputs(case, seed)
        return dict(case=case, net=net, f=f, u=u if kind == "train" else torch.empty_like(f))
    ps = [_setup(case, t) for t in range(_ntrees(case))]
    p = ps[0]
    st = dict(case=case, p=p, ps=ps, geom=solver.geometry_from_code(p["geom"]), bc=p["bc"])
    if kind == "photo":
        ctx = solver.Context.forest([(q["tree"], q["conn"]) for q in ps], p["M"])
        st["disc"] = [solver.HelmholtzDiscretization(2, 2, q["k2"]) for q in ps]
        st["s"] = [q["s"] for q in ps]
        host = solver.concat_fields([_host(_charge(q, seed if t < 3 else seed + t), 2, 1) for t, q in enumerate(ps)])
    else:
        ctx = solver.Context(p["tree"], p["conn"], p["M"])
        st["disc"] = solver.LaplacianDiscretization(p["D"], case.get("order", 2))
        st["s"] = p["s"]
        host = _host(_charge(p, seed), p["D"], 2 if kind == "dropin" else 1)
    st["ctx"] = ctx
    names = [("u", F64), ("b", F64)]
    names += [(k, F32) for k in ("e", "be", "re", "ue")] if case.get("form") == "mixed" else [("r", F64), ("u1", F64)]
    st.update({k: ctx.field(t) for k, t in names})
    if kind == "poisson":
        st["q"] = ctx.field(F64).upload(host)
    elif kind == "dropin":
        st["bh"], st["uh"] = host, np.zeros(host.shape, order="F")
        _restrict_host(st, seed)
    else:
        st["b"].upload(host)
    ctx.synchronize()
    return st


def _restrict_host(st, seed):
    """Covered cells of the host right-hand side: means of their children."""
    a, M = Forest(st["p"]), st["p"]["M"]
    b = a.split(_charge(st["p"], seed))
    a.restrict_all(b)
    v = a.join(b).cpu().numpy().transpose(2, 1, 0)
    st["bh"][2:2 + M, 2:2 + M, :] = v


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "poisson":
        solver.poisson_step(st["u"], st["b"], st["r"], st["u1"], st["s"], st["geom"], st["bc"], st["disc"],
                            poisson_iter=case["iters"], q=st["q"])
        return Resident(u=lambda: _read(st["u"]))
    if kind == "solve":
        # the last solve's right-hand sides on covered cells give way to the means
        solver.restrict_full(st["b"])
        if case["form"] == "fp64":
            n, hist = solver.solve(st["u"], st["b"], st["r"], st["u1"], st["s"], st["geom"], st["bc"], st["disc"],
                                   tol=TOL, guess=solver.GUESS_ZERO)
        else:
            n, hist = solver.solve_mixed(st["u"], st["b"], st["e"], st["be"], st["re"], st["ue"], st["s"], st["geom"],
                                         st["bc"], st["disc"], tol=TOL, inner_cycles=3, inner_first=2,
                                         guess=solver.GUESS_ZERO)
        return Resident(u=lambda: _read(st["u"]), cycles=n)
    if kind == "photo":
        solver.restrict_full(st["b"])
        if case["form"] == "fp64":
            n, hist = solver.solve_batched(st["u"], st["b"], st["r"], st["u1"], st["s"], st["geom"], st["bc"],
                                           st["disc"], tol=TOL, guess=solver.GUESS_ZERO)
        else:
            n, hist = solver.solve_mixed_batched(st["u"], st["b"], st["e"], st["be"], st["re"], st["ue"], st["s"],
                                                 st["geom"], st["bc"], st["disc"], tol=TOL, inner_cycles=2,
                                                 guess=solver.GUESS_ZERO)
        return Resident(u=lambda: _read(st["u"]), cycles=n)
    if kind == "dropin":
        st["u"].upload(st["uh"])
        st["b"].upload(st["bh"])
        solver.vcycle(st["u"], st["b"], st["r"], st["u1"], st["s"], geometry=st["geom"], bc=st["bc"],
                      lpldisc=st["disc"], ndown=2, ntop=4, nup=2)
        st["u"].download(st["uh"], bc=st["bc"])
        st["b"].download(st["bh"], bc=st["bc"])
        return {"u": st["uh"], "b": st["bh"]}
    if kind == "grid":
        solver.grid_solve(st["ctx"], case["D"], st["n"], st["s"], st["geom"], st["bc"], st["disc"], st["f"], st["u"],
                          case["grids"])
        return st["u"]
    if kind == "infer":
        st["net"].forward(st["f"], st["u"], case["batch"])
        return st["u"]
    st["net"].train_step(st["f"], st["u"], case["batch"], 1e-3)
    return Resident(params=lambda: st["net"].get_params())


def _conv_layers(D, widths):
    L = len(widths)
    out, cin = [], 8
    for l in range(L):
        out += [(l, cin, widths[l]), (l, widths[l], widths[l])]
        cin = widths[l]
    for l in range(L - 2, -1, -1):
        out += [(l + 1, widths[l + 1], widths[l]), (l, widths[l], widths[l])]
    return out + [(0, widths[0], 1)]


def work(case):
    """Each input read once and each output written once; the products and sums
    of the cycles a solve to 1e-8 takes (8 of FP64, 9 with the FP64 defects of
    the mixed form), of one V-cycle, of the axis transforms, of the convolutions."""
    kind = case["kind"]
    if kind == "grid":
        n = [case["n0"], case["n1"], case["n2"]][:case["D"]]
        v = case["grids"] * math.prod(n)
        return {"bytes": 16 * v, "flops": 4 * v * sum(n)}
    if kind in ("infer", "train"):
        par, _, widths = _weights(case)
        D, n = NETS[case["net"]]
        v = math.prod(n)
        fl = case["batch"] * sum(2 * 3 ** D * ci * co * (v >> (D * l)) for l, ci, co in _conv_layers(D, widths))
        if kind == "infer":
            return {"bytes": 8 * v * case["batch"] + 4 * par.size, "flops": fl}
        return {"bytes": 8 * v * case["batch"] + 24 * par.size, "flops": 3 * fl}
    cells = 0
    for t in range(_ntrees(case)):
        p = _setup(case, t)
        cells += p["tree"].nblocks() * p["M"] ** p["D"]
    D = 2 if kind == "photo" else case["D"]
    cyc = case["iters"] if kind == "poisson" else 1 if kind == "dropin" else 8 if case["form"] == "fp64" else 9
    # a V-cycle: four sweeps, a residual and its restriction, the transfers
    per = 4 * (4 * D + 5) + (4 * D + 4) + 3 + 2 * D + 6
    words = 3 if kind == "dropin" else 2
    w = 8 * words * cells * ((p["M"] + 4) / p["M"]) ** D if kind == "dropin" else 8 * words * cells
    return {"bytes": w, "flops": per * cells * cyc}


# ---- the same in 64 bits ----

class Forest:
    """One tree's levels as torch arrays [blocks, (z,) y, x] in `pairs` order,
    with the multigrid operations on lists of such arrays (one per level)."""

    def __init__(self, p):
        self.D, self.M, self.s = p["D"], p["M"], p["s"]
        D, M = self.D, self.M
        self.k2, self.geom = p["k2"], p["geom"]
        bc = np.asarray(p["bc"]).reshape((3,) * D, order="F")
        self.bcd = []
        for d in range(D):
            at = [1] * D
            lo, hi = list(at), list(at)
            lo[d], hi[d] = 0, 2
            self.bcd.append((float(bc[tuple(lo)]), float(bc[tuple(hi)])))
        self.root = p["root"]
        self.nblk = p["tree"].nblocks()
        self.co, self.id, self.nb, self.cf, self.par, self.sub = [], [], [], [], [], []
        maps = []
        for l, layer in enumerate(p["tree"]):
            co = torch.tensor([c for c, _ in layer.pairs], device=DEV).reshape(-1, D) - 1
            ext = [n << l for n in p["root"]]
            mp = torch.full([e + 2 for e in ext], -1, dtype=torch.int64, device=DEV)
            mp[tuple(co[:, d] + 1 for d in range(D))] = torch.arange(len(co), device=DEV)
            maps.append(mp)
            self.co.append(co)
            self.id.append(torch.tensor([b for _, b in layer.pairs], device=DEV, dtype=torch.int64) - 1)
            nb, cf = [], []
            for f in range(2 * D):
                q = co.clone()
                q[:, f >> 1] += 1 if f & 1 else -1
                j = mp[tuple(q[:, d] + 1 for d in range(D))]
                inside = (q[:, f >> 1] >= 0) & (q[:, f >> 1] < ext[f >> 1])
                k = torch.nonzero(inside & (j < 0)).reshape(-1)
                nb.append(j)
                qk = q[k]
                c = maps[l - 1][tuple((qk[:, d] >> 1) + 1 for d in range(D))] if l else k
                cf.append((k, c, sum((qk[:, d] & 1) << d for d in range(D)) if len(k) else k))
            self.nb.append(nb)
            self.cf.append(cf)
            if l:
                self.par.append(maps[l - 1][tuple((co[:, d] >> 1) + 1 for d in range(D))])
                self.sub.append(sum((co[:, d] & 1) << d for d in range(D)))
            else:
                self.par.append(None)
                self.sub.append(None)
        self.L = len(self.co)
        par = torch.arange(M, device=DEV)
        self.odd = (sum(par.reshape([M if a == d else 1 for a in range(D)]) for d in range(D)) + D) % 2 == 1

    def split(self, a):
        return [a[i].clone() for i in self.id]

    def join(self, lv):
        out = torch.zeros((self.nblk,) + lv[0].shape[1:], dtype=torch.float64, device=DEV)
        for i, a in zip(self.id, lv):
            out[i] = a
        return out

    def zeros(self):
        return [torch.zeros((len(i),) + (self.M,) * self.D, dtype=torch.float64, device=DEV) for i in self.id]

    def slabs(self):
        return [[torch.zeros((len(k),) + (self.M,) * (self.D - 1), dtype=torch.float64, device=DEV)
                 for k, _, _ in cf] for cf in self.cf]

    def padded(self, u, l, slab):
        """u[l] with one layer of face ghosts: copies, mirrors, the slabs."""
        D, M = self.D, self.M
        P = torch.nn.functional.pad(u[l], (1, 1) * D)
        mid = slice(1, M + 1)
        for f in range(2 * D):
            ax, hi = D - (f >> 1), f & 1
            v = u[l].select(ax, M - 1 if hi else 0) * self.bcd[f >> 1][hi]
            j = self.nb[l][f]
            k = torch.nonzero(j >= 0).reshape(-1)
            v[k] = u[l].select(ax, 0 if hi else M - 1)[j[k]]
            if slab is not None and len(self.cf[l][f][0]):
                v[self.cf[l][f][0]] = slab[l][f]
            at = [slice(None)] + [mid] * D
            at[ax] = (M + 1) if hi else 0
            P[tuple(at)] = v
        return P

    def prolong(self, P, sub):
        """The fine cells over subblock `sub` of each padded block of P."""
        D, M = self.D, self.M
        h = M // 2
        out = torch.empty((len(P),) + (M,) * D, dtype=torch.float64, device=DEV)
        w0 = 0.5 if D == 2 else 0.25
        for code in range(1 << D):
            k = torch.nonzero(sub == code).reshape(-1)
            if not len(k):
                continue
            A = P[k]
            o = torch.empty((len(k),) + (M,) * D, dtype=torch.float64, device=DEV)
            base = [1 + h * ((code >> d) & 1) for d in range(D)]

            def win(shift):
                return A[(slice(None),) + tuple(slice(base[d] + shift[d], base[d] + shift[d] + h)
                                                for d in range(D - 1, -1, -1))]
            for ii in range(1 << D):
                v = w0 * win([0] * D)
                for d in range(D):
                    sh = [0] * D
                    sh[d] = 2 * ((ii >> d) & 1) - 1
                    v = v + 0.25 * win(sh)
                o[(slice(None),) + tuple(slice((ii >> d) & 1, None, 2) for d in range(D - 1, -1, -1))] = v
            out[k] = o
        return out

    def fill(self, u, l, slab):
        """The coarse-fine ghosts of level l from level l - 1."""
        if l == 0 or slab is None or not any(len(k) for k, _, _ in self.cf[l]):
            return
        P = self.padded(u, l - 1, slab)
        for f in range(2 * self.D):
            k, c, sub = self.cf[l][f]
            for a in range(0, len(k), 4096):
                e = slice(a, a + 4096)
                slab[l][f][e] = self.prolong(P[c[e]], sub[e]).select(self.D - (f >> 1), 0 if f & 1 else self.M - 1)

    def restrict(self, u, l, src=None):
        """Children's means into u[l - 1] (of src[l] where given)."""
        a = (u if src is None else src)[l]
        D, h = self.D, self.M // 2
        for d in range(1, D + 1):
            a = a.unflatten(d, (self.M // 2, 2)).sum(d + 1)
        a = a / (1 << D)
        for code in range(1 << D):
            k = torch.nonzero(self.sub[l] == code).reshape(-1)
            at = tuple(slice(h * ((code >> d) & 1), h * ((code >> d) & 1) + h) for d in range(D - 1, -1, -1))
            u[l - 1][(self.par[l][k],) + at] = a[k]

    def restrict_all(self, u):
        for l in range(self.L - 1, 0, -1):
            self.restrict(u, l)

    def apply(self, u, l, slab, sl):
        """(L u on level l, its centre coefficient)"""
        D, M = self.D, self.M
        P = self.padded(u, l, slab)
        cc = -2.0 * D - (sl * self.k2 if self.k2 is not None else 0.0)
        v = cc * u[l]
        for d in range(D):
            ax = D - d
            lo, hi = ([slice(None)] + [slice(1, M + 1)] * D for _ in range(2))
            lo[ax], hi[ax] = slice(0, M), slice(2, M + 2)
            if self.geom == d + 1:
                J = (self.co[l][:, d:d + 1] * M + torch.arange(1, M + 1, device=DEV)).double()
                J = J.reshape([len(J)] + [M if a == ax else 1 for a in range(1, D + 1)])
                v = v + (2 * J - 2) / (2 * J - 1) * P[tuple(lo)] + 2 * J / (2 * J - 1) * P[tuple(hi)]
            else:
                v = v + P[tuple(lo)] + P[tuple(hi)]
        return v, cc

    def smooth(self, u, b, l, slab, n):
        sl = self.s / 4 ** l
        for _ in range(n):
            for first in (True, False):
                Lu, cc = self.apply(u, l, slab, sl)
                v = u[l] - (Lu + sl * b[l]) / cc
                u[l] = torch.where(self.odd if first else ~self.odd, v, u[l])

    def top(self, u, b, slab, exact):
        if not exact:
            return self.smooth(u, b, 0, slab, 4)
        D, M = self.D, self.M
        n = [r * M for r in self.root]
        g = torch.empty(tuple(reversed(n)), dtype=torch.float64, device=DEV)
        cell = [(self.co[0][:, d:d + 1] * M + torch.arange(M, device=DEV)).reshape(
            [-1] + [M if a == D - 1 - d else 1 for a in range(D)]) for d in range(D)]
        at = tuple(cell[d] for d in range(D - 1, -1, -1))
        g[at] = -self.s * b[0]
        x = _level1(g[None], n, self.geom, self.bcd, -self.s * self.k2 if self.k2 is not None else 0.0)
        u[0] = x[0][at]

    def vcycle(self, u, b, slab, exact):
        r, u1, s1 = self.zeros(), [None] * self.L, self.slabs()
        for l in range(self.L - 1, 0, -1):
            sl = self.s / 4 ** l
            self.smooth(u, b, l, slab, 2)
            r[l] = -(b[l] + self.apply(u, l, slab, sl)[0] / sl)
            self.restrict(u, l)
            self.fill(u, l - 1, slab)
            u1[l - 1] = u[l - 1].clone()
            self.restrict(r, l)
            Lu, _ = self.apply(u, l - 1, slab, 4 * sl)
            new = -(r[l - 1] + Lu / (4 * sl))
            under = torch.zeros_like(b[l - 1], dtype=torch.bool)
            h = self.M // 2
            for code in range(1 << self.D):
                k = torch.nonzero(self.sub[l] == code).reshape(-1)
                at = tuple(slice(h * ((code >> d) & 1), h * ((code >> d) & 1) + h) for d in range(self.D - 1, -1, -1))
                under[(self.par[l][k],) + at] = True
            b[l - 1] = torch.where(under, new, b[l - 1])
        self.top(u, b, slab, exact)
        for l in range(1, self.L):
            u1[l - 1] = u[l - 1] - u1[l - 1]
            self.fill(u1, l - 1, s1)
            P = self.padded(u1, l - 1, s1)
            for a in range(0, len(self.co[l]), 16384):
                e = slice(a, a + 16384)
                u[l][e] += self.prolong(P[self.par[l][e]], self.sub[l][e])
            self.fill(u, l, slab)
            self.smooth(u, b, l, slab, 2)
            self.fill(u, l, slab)


def _out(a, G=0):
    """[blocks, (z,) y, x] as a host array in the layout of the device fields' reads."""
    return _host(a, a.dim() - 1, G)


def _exact_net(case, seed):
    """(FP64 parameters, the network's prediction and loss as functions)."""
    par, c_out, widths = _weights(case)
    D, n = NETS[case["net"]]
    n = n[:D]
    f, u = _net_inputs(case, seed)
    B = len(f)
    grid = (B,) + tuple(reversed(n))
    f, u = f.double().reshape(grid), u.double().reshape(grid)
    scale = f.reshape(B, -1).abs().amax(1)
    scale = torch.where(scale > 0, scale, torch.ones_like(scale)).reshape([B] + [1] * D)
    x = torch.zeros(grid + (8,), dtype=torch.float64, device=DEV)
    x[..., 0] = f / scale
    for d in range(D):
        c = 2 * (torch.arange(n[d], device=DEV, dtype=torch.float64) + 0.5) / n[d] - 1
        x[..., 1 + d] = c.reshape([1] + [n[d] if a == D - 1 - d else 1 for a in range(D)])

    def conv(x, p):
        W, b = p
        xp = torch.nn.functional.pad(x, (0, 0) + (1, 1) * D)
        out = b
        for t in range(3 ** D):
            off = [(t // 3 ** d) % 3 for d in range(D)]
            sl = (slice(None),) + tuple(slice(off[d], off[d] + n_) for d, n_ in
                                        zip(range(D - 1, -1, -1), x.shape[1:-1])) + (slice(None),)
            out = out + xp[sl] @ W[:, t, :].T
        return out

    def pool(x):
        for d in range(1, D + 1):
            x = x.unflatten(d, (x.shape[d] // 2, 2)).mean(d + 1)
        return x

    def up(x):
        for d in range(1, D + 1):
            x = x.repeat_interleave(2, d)
        return x

    def predict(flat):
        P, o = [], 0
        for _, ci, co in _conv_layers(D, widths):
            m = co * 3 ** D * ci
            P.append((flat[o:o + m].reshape(co, 3 ** D, ci), flat[o + m:o + m + co]))
            o += m + co
        P, L, E, v = iter(P), len(widths), [], x
        for l in range(L):
            v = pool(v) if l else v
            v = conv(conv(v, next(P)).relu(), next(P)).relu()
            E.append(v)
        for l in range(L - 2, -1, -1):
            v = conv(up(conv(v, next(P))) + E[l], next(P)).relu()
        return conv(v, next(P))[..., 0]

    return par, lambda q: predict(q) * scale * c_out, lambda q: ((predict(q) - u / (scale * c_out)) ** 2).mean()


def _first_weights(case, seed):
    """He-normal weights and zero biases: where a training begins."""
    D, _ = NETS[case["net"]]
    r = np.random.default_rng(seed)
    out = []
    for _, ci, co in _conv_layers(D, _weights(case)[2]):
        out += [r.normal(0, math.sqrt(2 / (3 ** D * ci)), co * 3 ** D * ci), np.zeros(co)]
    return np.concatenate(out).astype(np.float32)


def exact(case, seed):
    kind = case["kind"]
    if kind == "grid":
        D = case["D"]
        n = [case["n0"], case["n1"], case["n2"]][:D]
        s = (1e-2 / n[0]) ** 2 * configs.ELEMENTARY_CHARGE / configs.EPSILON_0
        f = -s * _grid_charges(n, case["geom"], case["grids"], seed, 0.05)
        bcd = _grid_bc(D, case["geom"])
        return _level1(f.reshape((-1,) + tuple(reversed(n))), n, case["geom"], bcd).reshape(f.shape)
    if kind == "infer":
        par, predict, _ = _exact_net(case, seed)
        with torch.no_grad():
            y = predict(torch.tensor(par, dtype=torch.float64, device=DEV))
        return y.reshape(y.shape[0], -1)
    if kind == "train":
        _, _, loss = _exact_net(case, seed)
        q = torch.tensor(_first_weights(case, seed), dtype=torch.float64, device=DEV, requires_grad=True)
        g, = torch.autograd.grad(loss(q), q)
        return {"params": (q.detach() - 1e-3 * g / (g.abs() + 1e-8)).cpu().numpy()}
    if kind == "poisson" and case["order"] == 4:
        return None  # its ghost frames' order of filling is the library's alone
    done = []
    for t in range(_ntrees(case)):
        p = _setup(case, t)
        a = Forest(p)
        u, slab = a.zeros(), a.slabs()
        b = a.split(_charge(p, seed if t < 3 else seed + t))
        a.restrict_all(b)
        if kind == "poisson":
            for _ in range(case["iters"]):
                for l in range(1, a.L):
                    a.fill(u, l, slab)
                a.vcycle(u, b, slab, False)
        elif kind == "dropin":
            a.vcycle(u, b, slab, False)
            return {"u": _ghosts(a, u, slab), "b": _ghosts(a, b, None)}
        else:
            for _ in range(14):  # a tenth of the error stays after each: to rounding
                a.vcycle(u, b, slab, True)
        done.append(a.join(u))
    v = _out(torch.cat(done))
    return {"u": v} if kind == "poisson" else {"u": v, "cycles": None}


def _ghosts(a, u, slab):
    """Host arrays with two ghost layers of which the faces' inner one is filled."""
    M = a.M
    out = torch.zeros((a.nblk, M + 2, M + 2), dtype=torch.float64, device=DEV)
    for l in range(a.L):
        out[a.id[l]] = a.padded(u, l, slab if slab is not None else a.slabs())
    return _host(out, 2, 1)
