"""Batches whose tensors pass 2^31 values, where pooling, upsampling and their
adjoints index in 64 bits: every grid of a batch of 16 256^3 grids equals the
prediction of that grid alone (which indexes in 32 bits), bit for bit; and the
gradient of 16 equal grids that of one. The latter's gradients at the layers are
those of one grid over 16, exactly (a power of two), so only the FP32 sums over 16
times as many voxels differ: 2e-2 per convolution, as between the network and its
restatement."""

import numpy as np
import pytest

from srmg import solver

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

N, B = 256, 16
WIDTHS = (8, 8)


def _need(gib):
    free, _ = torch.cuda.mem_get_info()
    if free < gib * 2 ** 30:
        pytest.skip(f"needs {gib} GiB of GPU memory")


def test_large_batch_equals_single_grids():
    _need(80)
    print(f"network on {B} grids of {N}^3", flush=True)
    net = solver.UNet(3, (N,) * 3, 2, WIDTHS, seed=3)
    g = torch.Generator(device="cuda").manual_seed(1)
    f = torch.randn(B, N ** 3, device="cuda", generator=g)
    out = torch.empty_like(f)
    torch.cuda.synchronize()
    net.forward(f, out, B)
    net.synchronize()
    assert torch.isfinite(out).all()
    for k in (0, 7, B - 1):
        one = torch.empty_like(f[k])
        net.forward(f[k].contiguous(), one, 1)
        net.synchronize()
        assert torch.equal(out[k], one), f"grid {k}"


def test_large_batch_gradient():
    _need(80)
    print(f"gradient on {B} grids of {N}^3", flush=True)
    net = solver.UNet(3, (N,) * 3, 2, WIDTHS, seed=4)
    g = torch.Generator(device="cuda").manual_seed(2)
    f, u = torch.randn(1, N ** 3, device="cuda", generator=g), torch.randn(1, N ** 3, device="cuda", generator=g)
    torch.cuda.synchronize()
    loss1, g1 = net.loss_grad(f, u, 1)
    fb, ub = f.repeat(B, 1), u.repeat(B, 1)
    torch.cuda.synchronize()
    loss, gb = net.loss_grad(fb, ub, B)
    assert abs(loss - loss1) < 2e-3 * loss1
    widths, o = [(8, 8), (8, 8), (8, 8), (8, 8), (8, 8), (8, 8), (8, 1)], 0
    for k, (ci, co) in enumerate(widths):
        m = co * 27 * ci + co
        rel = np.linalg.norm(gb[o:o + m] - g1[o:o + m]) / np.linalg.norm(g1[o:o + m])
        print(f"  conv {k} ({ci}->{co}): {rel:.2e}")
        assert rel < 2e-2
        o += m
