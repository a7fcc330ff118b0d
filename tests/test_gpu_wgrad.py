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
