"""Host fields whose block ids are scattered over more places than the tree has
blocks (refinement frees ids and takes others): cells and ghosts against the
records, other blocks' places untouched, also after the context took another
tree. Blocks large and small, in few pieces and in many."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")  # noqa: F841  (torch's HIP runtime first)

from srmg import solver
from srmg.solver import F32, F64
from srmg.tree import boundaryconditions, connectivity, refined_tree
from test_gpu_host_fields import BCS, expected

pytestmark = pytest.mark.gpu


def _scattered(D, root, levels, width, rng):
    """A tree whose ids are drawn from 1 .. about `width` times its blocks."""
    tree = refined_tree(D, root, levels, lambda l, c: np.all(c <= 1, axis=1) | (c[:, 0] == 2))
    n = tree.nblocks() * width + 3
    ids = rng.choice(n, size=tree.nblocks(), replace=False) + 1
    if width == 1:
        ids.sort()  # runs with gaps
    for layer in tree:
        items = [(c, int(ids[b - 1])) for c, b in layer.index.items()]
        layer.index, layer.coord = dict(items), {b: c for c, b in items}
    tree.sync()
    return tree, connectivity(tree), n


@pytest.mark.parametrize("D,M,root,levels", [(2, 16, (2, 3), 3), (2, 8, (40, 50), 2), (3, 8, (10, 6, 9), 2),
                                             (3, 16, (2, 1, 3), 2)])
@pytest.mark.parametrize("width", [1, 2, 9])
def test_scattered_block_ids(D, M, root, levels, width):
    print(f"host ids D={D} M={M} root={root} width={width}", flush=True)
    rng = np.random.default_rng(17 * D + M + width)
    bc = np.asarray(boundaryconditions(BCS[D]), np.int8).ravel()
    ctx = None
    for _ in range(2):  # the second tree replaces the first
        tree, conn, n = _scattered(D, root, levels, width, rng)
        if ctx is None:
            ctx = solver.Context(tree, conn, M, nblocks=n)
        else:
            ctx.regrid(tree, conn, nblocks=n)
        for dtype, hin, gin, hout, gout in [(F64, np.float64, 2, np.float64, 2), (F32, np.float64, 3, np.float32, 1),
                                            (F64, np.float32, 1, np.float64, 0)]:
            host = np.asfortranarray(rng.normal(size=(M + 2 * gin,) * D + (n,)).astype(hin))
            f = ctx.field(dtype).upload(host)
            seen = host.astype(np.float32) if dtype == F32 else host  # what the device holds
            out = np.full((M + 2 * gout,) * D + (n,), 7.25, hout, order="F")
            want = expected((tree, conn, D, M, gout), seen, out.copy(order="F"), gout, bc)
            f.download(out, bc=bc)
            np.testing.assert_array_equal(out, want)
            f.close()
