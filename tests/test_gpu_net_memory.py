"""What the network allocates: an inference nothing that only training needs."""
import numpy as np
import pytest
import torch

from karman_taichi_amd import _lib
from karman_taichi_amd._lib import ptr
from oracle import unet
from unet_systems import small_system

pytestmark = pytest.mark.gpu
MB = 1 << 20


def held(f):
    """Device memory f() leaves allocated, beyond torch's own."""
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    f()
    torch.cuda.synchronize()
    return before - torch.cuda.mem_get_info()[0]


def test_inference_holds_no_training_memory(dev):
    """64 x 32 cells: activations of a few hundred bytes per cell (1 MB) and
    8 MB of partial sums.  Training adds the 128 MB of its partial sums, once,
    and a context that has inferred before gives the same gradients."""
    nx, ny = 64, 32
    coef, r = small_system(5, nx=nx, ny=ny)
    params = torch.tensor(unet.init_params(3), device=dev)
    c, rt = torch.tensor(coef, device=dev), torch.tensor(r, device=dev)
    c32, r32 = c.float(), rt.float()
    z = torch.empty_like(rt)
    grads = [torch.empty_like(params) for _ in range(2)]
    stream = torch.cuda.current_stream(dev).cuda_stream
    ctxs = [_lib.Context(torch.cuda.current_device(), stream) for _ in range(2)]

    def infer(k):
        ctxs[k].call("km_unet_apply", ptr(params), nx + 2, ny + 2, ptr(c), ptr(rt), ptr(z))

    def train(k):
        ctxs[k].call("km_unet_loss_grad", ptr(params), 1, nx + 2, ny + 2, ptr(c32), ptr(r32), None, ptr(grads[k]),
                     None)

    try:
        train(1)    # the HIP runtime's own memory for these kernels comes with the first context
        infer(1)
        used = held(lambda: infer(0))
        print(f"inference {used / MB:.0f} MB")
        assert used < 32 * MB
        used = held(lambda: train(0))
        print(f"training after it {used / MB:.0f} MB more")
        assert used < 160 * MB
        assert held(lambda: (infer(0), train(0))) == 0
        torch.cuda.synchronize()
        assert torch.equal(grads[0], grads[1]) and bool(torch.isfinite(grads[0]).all())
        assert np.count_nonzero(grads[0].cpu().numpy()) > 0
    finally:
        for ctx in ctxs:
            ctx.close()


def test_more_pixels_than_the_kernels_count_are_refused(dev):
    """64 images of 8192 x 8192 pixels are 2^32: refused by the size, before
    anything is allocated or read."""
    params = torch.tensor(unet.init_params(3), device=dev)
    ctx = _lib.Context(torch.cuda.current_device(), torch.cuda.current_stream(dev).cuda_stream)
    try:
        with pytest.raises(_lib.KarmanError, match="too many"):
            ctx.call("km_unet_loss_grad", ptr(params), 64, 8194, 8194, ptr(params), ptr(params), None, ptr(params), None)
    finally:
        ctx.close()
