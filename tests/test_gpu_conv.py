"""The network's convolutions at the edges of their tiles (16 columns by 4 to 16
rows of pixels at each of the four levels): images smaller than a tile, exactly
one, one and a remainder in each direction, and a level of a single pixel.

Against the oracle with BF16 rounding at the kernels' rounding points.  The
bound on the relative 2-norm error, 1e-2, is that of the forward test at
30 x 22: another order of the FP32 sums flips single BF16 roundings (2^-9) of
some activations, and the seven layers' flips together stay below five of those.
"""
import numpy as np
import pytest
import torch

from karman_taichi_amd import _lib
from karman_taichi_amd._lib import ptr
from oracle import unet
from unet_systems import small_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(8, 8), (16, 16), (9, 130), (136, 24), (65, 33)])
def test_forward_at_tile_edges(nx, ny, dev):
    coef, r = (np.asarray(a, np.float32).astype(np.float64) for a in small_system(70, nx=nx, ny=ny))
    params = unet.init_params(6)
    params[unet.param_slices()[0]["out.b"][0]] = 0.05
    pt, ct, rt = (torch.tensor(a, device=dev) for a in (params, coef, r))
    zt = torch.empty_like(rt)
    _lib.context_for(dev).call("km_unet_apply", ptr(pt), nx + 2, ny + 2, ptr(ct), ptr(rt), ptr(zt))
    z = zt.cpu().numpy()
    zo = unet.apply(params.astype(np.float64), coef, r, bf=True)
    err = np.linalg.norm(z - zo) / np.linalg.norm(zo)
    print(f"{nx}x{ny}: {err:.1e}")
    assert err < 1e-2


def test_forward_in_place(dev):
    """The output may be the right-hand side's own buffer."""
    coef, r = small_system(71, nx=65, ny=33)
    pt = torch.tensor(unet.init_params(6), device=dev)
    ct, rt = torch.tensor(coef, device=dev), torch.tensor(r, device=dev)
    zt = torch.empty_like(rt)
    ctx = _lib.context_for(dev)
    ctx.call("km_unet_apply", ptr(pt), 67, 35, ptr(ct), ptr(rt), ptr(zt))
    ctx.call("km_unet_apply", ptr(pt), 67, 35, ptr(ct), ptr(rt), ptr(rt))
    assert torch.equal(rt, zt)
