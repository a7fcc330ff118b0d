"""Weight and bias gradients of the network at sizes where the pixel chunks of
the weight-gradient kernel end: one chunk of 64 pixels, images whose rows are
shorter or longer than a chunk, several images per chunk (the coarsest level of
the smallest one is a single pixel).  Against the oracle with BF16 rounding at
the kernels' rounding points; the bound on each parameter's relative 2-norm
error, 3e-2, is that of the gradient test at 30 x 22: BF16 keeps 8 bits, so a
value is off by at most 2^-9, and a handful of layers' roundings in a row stay
below ten of those.
"""
import numpy as np
import pytest
import torch

from karman_taichi_amd import learned
from oracle import unet
from unet_systems import small_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,B", [(8, 8, 1), (8, 8, 5), (9, 71, 2), (40, 9, 3)])
def test_gradients_at_chunk_edges(nx, ny, B, dev):
    systems = [small_system(40 + k, nx=nx, ny=ny) for k in range(B)]
    coefs = np.stack([c for c, _ in systems]).astype(np.float32)
    rs = np.stack([r for _, r in systems]).astype(np.float32)
    params = unet.init_params(11)
    net = learned.UNetPreconditioner(params=params, device=dev)
    _, grad = net.loss_grad(torch.tensor(coefs, device=dev), torch.tensor(rs, device=dev))
    g = grad.cpu().numpy().astype(np.float64)
    _, go, _ = unet.loss_and_grad(params.astype(np.float64), coefs.astype(np.float64), rs.astype(np.float64), bf=True)
    for name, (o, shape) in unet.param_slices()[0].items():
        m = int(np.prod(shape))
        a, b = g[o:o + m], go[o:o + m]
        err = np.linalg.norm(a - b) / np.linalg.norm(b)
        print(f"{nx}x{ny} x {B} {name}: {err:.1e}")
        assert err < 3e-2, name


@pytest.mark.parametrize("nx,ny", [(1280, 192), (328, 72), (96, 24)])
def test_gradients_of_copies_equal_those_of_one(nx, ny, dev):
    """Four copies of a system have the gradient of one (the loss is a mean, its
    factor 1/4 exact) with the pixels shared out differently among the
    workgroups: 32 to 576 each, and at 1280 x 192 shares of 96 pixels, a chunk
    and a half.  An FP32 sum of 576 terms is off by at most 576 x 2^-24 = 3.4e-5
    of the sum of their magnitudes; the bound on the difference, 1e-4 of the
    layer's largest weight gradient, is that with room for terms that cancel
    threefold."""
    coef, r = small_system(7, nx=nx, ny=ny)
    params = unet.init_params(11)
    net = learned.UNetPreconditioner(params=params, device=dev)
    grads = []
    for B in (1, 4):
        c = torch.tensor(np.stack([coef] * B).astype(np.float32), device=dev)
        rt = torch.tensor(np.stack([r] * B).astype(np.float32), device=dev)
        _, g = net.loss_grad(c, rt)
        grads.append(g.cpu().numpy().astype(np.float64).copy())
    for name, (o, shape) in unet.param_slices()[0].items():
        m = int(np.prod(shape))
        a, b = grads[0][o:o + m], grads[1][o:o + m]
        err = np.abs(a - b).max() / np.abs(a).max()
        print(f"{nx}x{ny} {name}: {err:.1e}")
        assert err < 1e-4, name
