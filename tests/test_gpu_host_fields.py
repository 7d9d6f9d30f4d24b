"""Host fields to the device and back in pieces: every cell and ghost that the
host layout holds, against the records, bit for bit (FP32 on either side rounds
once). The sizes cover one piece, several, and enough for the threads that
place the pieces; ghost depths 0 to 3; block ids that no block has."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")  # noqa: F841  (torch's HIP runtime first)

from srmg import solver
from srmg.solver import F32, F64
from srmg.tree import boundaryconditions, connectivity, refined_tree

pytestmark = pytest.mark.gpu

# D, M, root, levels refined around the first corner
TREES = [(2, 16, (2, 3), 3), (2, 8, (40, 50), 2), (3, 8, (3, 2, 4), 2), (3, 8, (10, 12, 9), 2), (3, 16, (2, 1, 3), 2)]
BCS = {2: ((1, -1), (-1, 1)), 3: ((1, -1), (-1, 1), (1, -1))}


def expected(p, host, out, G, bc):
    """`out` after a download of what an upload of `host` left on the device."""
    tree, conn, D, M, Gi = p
    g0 = (host.shape[0] - M) // 2
    assert Gi == G
    def box(G, face, inner):
        # the cells of a face layer: the ghosts, or the valid cells at it
        return tuple(slice(G, G + M) if f == 0 else
                     ((slice(G, G + 1) if f < 0 else slice(G + M - 1, G + M)) if inner else
                      (slice(G - 1, G) if f < 0 else slice(G + M, G + M + 1))) for f in face)
    v0, v = (slice(g0, g0 + M),) * D, (slice(G, G + M),) * D
    blocks = np.array([b for layer in tree for _, b in layer.pairs]) - 1
    t = out.dtype.type
    out[v + (blocks,)] = host[v0 + (blocks,)].astype(t)
    if G == 0:
        return out
    for l in range(len(tree)):
        for r in conn.neighbor[l]:
            face = tuple(r[2:2 + D])  # `to` lies on side `face` of `from`
            back = tuple(-f for f in face)
            out[box(G, back, False) + (r[1] - 1,)] = host[box(g0, face, True) + (r[0] - 1,)].astype(t)
        for r in conn.boundary[l]:
            face = tuple(r[1:1 + D])
            if bc is not None:
                sign = bc[sum((f + 1) * 3 ** d for d, f in enumerate(face))]
                out[box(G, face, False) + (r[0] - 1,)] = t(sign) * host[box(g0, face, True) + (r[0] - 1,)].astype(t)
        for r in conn.refboundary[l]:
            face = tuple(r[2:2 + D])
            out[box(G, face, False) + (r[0] - 1,)] = host[box(g0, face, False) + (r[0] - 1,)].astype(t)
    return out


@pytest.mark.parametrize("D,M,root,levels", TREES)
def test_upload_and_download_follow_the_records(D, M, root, levels):
    print(f"host fields D={D} M={M} root={root}", flush=True)
    tree = refined_tree(D, root, levels, lambda l, c: np.all(c <= 1, axis=1) | (c[:, 0] == 2))
    conn = connectivity(tree)
    nblocks = tree.nblocks() + 5  # ids that no block has
    bc = np.asarray(boundaryconditions(BCS[D]), np.int8).ravel()
    ctx = solver.Context(tree, conn, M, nblocks=nblocks)
    rng = np.random.default_rng(D * 100 + M)
    for dtype, hin, gin, hout, gout in [(F64, np.float64, 2, np.float64, 2), (F64, np.float64, 1, np.float64, 0),
                                        (F32, np.float64, 3, np.float32, 1), (F64, np.float32, 1, np.float64, 3)]:
        host = np.asfortranarray(rng.normal(size=(M + 2 * gin,) * D + (nblocks,)).astype(hin))
        f = ctx.field(dtype).upload(host)
        seen = host.astype(np.float32) if dtype == F32 else host  # what the device holds
        for with_bc in (True, False):
            out = np.full((M + 2 * gout,) * D + (nblocks,), 7.25, hout, order="F")
            want = expected((tree, conn, D, M, gout), seen, out.copy(order="F"), gout, bc if with_bc else None)
            f.download(out, bc=bc if with_bc else None)
            np.testing.assert_array_equal(out, want)
        f.close()
