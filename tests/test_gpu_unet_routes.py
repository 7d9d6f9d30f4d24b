"""The routes of the network's convolutions and weight gradients by grid size:
ragged tiles on either side of the share of a tile that a grid must fill, small
grids in large batches (gathered without a split of K), and rows too wide for
the weight gradients' LDS. Tolerances as in test_gpu_unet_tiles.py, for the same
reason."""

import os
import sys

import numpy as np
import pytest

from srmg import solver

sys.path.insert(0, os.path.join(os.path.dirname(__file__), "..", "oracle"))
import unet_ref as U  # noqa: E402

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

CASES = [
    (2, (60, 28), (8, 16), 40),      # 8 and 16 channels, 82% of ragged 2D tiles
    (2, (28, 30), (32, 16), 80),     # 32 channels, 82%
    (3, (14, 6, 6), (32, 8), 132),   # 32 channels, 49%
    (3, (6, 6, 6), (16, 8), 304),    # 21%: gathered
    (2, (18, 18), (8, 8), 204),      # 32%: gathered
    (2, (1024, 16), (8, 16), 5),     # one row of 1024 cells is too wide for the weight gradients' LDS
]


@pytest.mark.parametrize("D,n,widths,B", CASES)
def test_routes_match_cpu_restatement(D, n, widths, B):
    print(f"routes D={D} n={n} widths={widths} batch={B}", flush=True)
    rng = np.random.default_rng(5)
    net = solver.UNet(D, n, len(widths), widths)
    p = U.he_params(D, widths, rng, np.float32)
    net.set_params(p)
    net.output_scale = 5.0
    shape = (B,) + tuple(reversed(n))
    f, u = U.smooth_field(rng, shape), U.smooth_field(rng, shape) * 8.0
    fd, ud = (torch.tensor(a, dtype=torch.float32, device="cuda") for a in (f, u))
    out = torch.empty_like(fd)
    net.forward(fd, out, B)
    y, ca = U.forward(p.astype(np.float64), f, D, widths)
    ref = y * ca["scale"].reshape((B,) + (1,) * D) * 5.0
    assert np.max(np.abs(out.cpu().numpy() - ref)) < 3e-2 * np.max(np.abs(ref))
    loss, g = net.loss_grad(fd, ud, B)
    rloss, rg = U.loss_and_grad(p.astype(np.float64), f, u, 5.0, D, widths, bf16=True)
    assert abs(loss - rloss) < 2e-3 * rloss
    o = 0
    for k, (_, ci, co, _) in enumerate(U.layer_specs(widths)):
        m = co * 3 ** D * ci + co
        rel = np.linalg.norm(g[o:o + m] - rg[o:o + m]) / np.linalg.norm(rg[o:o + m])
        print(f"  conv {k} ({ci}->{co}): {rel:.2e}")
        assert rel < 2e-2
        o += m
