"""The network's LDS-tiled convolutions and weight gradients where tiles do not
fit the grid: extents that are no multiple of a tile (and of 8), grids smaller
than one tile, every channel count, batches on both sides of the split of the
K loop. Tolerances as in test_gpu_guess.py, for the same reason (BF16 stores,
FP32 accumulation in another order): loss 2e-3 and gradients 2e-2 per
convolution against the restatement that rounds at the same points, outputs
3e-2 in the max-norm against the exact one."""

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
    (2, (36, 20), (8, 16), 100),           # ragged in both dimensions
    (3, (20, 12, 28), (16, 32, 64), 12),   # ragged in 3D, rows of 5 voxels at the coarse level
    (3, (8, 4, 4), (32, 16), 520),         # grids smaller than a tile
    (2, (64, 32), (64, 8), 33),            # 64 channels on the unsplit path
    (3, (4, 4, 4), (8, 8), 1),             # the smallest grid
]


@pytest.mark.parametrize("D,n,widths,B", CASES)
def test_tiles_match_cpu_restatement(D, n, widths, B):
    print(f"tiles D={D} n={n} widths={widths} batch={B}", flush=True)
    rng = np.random.default_rng(3)
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
