"""Solves of systems whose rows of 255 and 256 cells, or of a few segments of
that length, do not fit the iteration kernels' tiles as one segment.

Against the direct solution: the error is at most cond(A) < 1e4 times the true
residual (rows sum to 0.01 or more and aP <= 7), eps = 1e-10, and the plain
solves, which stop on the recursive residual, may end at ten times eps.
"""
import ctypes

import numpy as np
import pytest
import torch

from karman_taichi_amd import _lib
from karman_taichi_amd._lib import KmSolveInfo, ptr
from oracle import krylov
from test_gpu_one_launch import EPS, system

pytestmark = pytest.mark.gpu

FLAGS = {"km_bicgstab": 0, "km_cg": 0, "km_bicgstab_noalloc": 0, "from_x": _lib.KM_FLAG_X0 | _lib.KM_FLAG_TRUE,
         "mixed": _lib.KM_FLAG_MIXED, "smooth": _lib.KM_FLAG_SMOOTH,
         "coarse": _lib.KM_FLAG_COARSE | _lib.KM_FLAG_SYMMETRIC}


@pytest.mark.parametrize("NY", [254, 255, 256, 257, 510, 512, 768, 1280])
@pytest.mark.parametrize("entry", list(FLAGS))
@pytest.mark.parametrize("launches", [False, True])
def test_rows_of_whole_segments(NY, entry, launches, dev):
    NX = 21
    coef, b = system(NX, NY, NY, 0.5)
    c, bt = torch.tensor(coef, device=dev), torch.tensor(b, device=dev)
    x, info = torch.zeros_like(bt), KmSolveInfo()
    ctx = _lib.Context(torch.cuda.current_device(), torch.cuda.current_stream(dev).cuda_stream)
    try:
        if launches:
            ctx.call("km_one_launch_give_up", 2)
        if entry in ("smooth", "coarse"):
            ctx.call("km_fbicgstab", NX, NY, ptr(c), ptr(bt), ptr(x), EPS, 0, FLAGS[entry], None, ctypes.byref(info))
        else:
            name = entry if entry.startswith("km_") else "km_bicgstab"
            ctx.call(name, NX, NY, ptr(c), ptr(bt), ptr(x), EPS, 0, FLAGS[entry], ctypes.byref(info))
        torch.cuda.synchronize()
    finally:
        ctx.close()
    xd = krylov.direct_solve(coef, b)
    err = np.linalg.norm(x.cpu().numpy() - xd) / np.linalg.norm(xd)
    print(f"{entry} {b.shape}: {info.iterations} it, true residual {info.rel_resid_true:.1e}, error {err:.1e}")
    assert info.status == _lib.KM_OK
    assert info.rel_resid_true < 10 * EPS
    assert err <= 1e5 * EPS
