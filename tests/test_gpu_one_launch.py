"""The preconditioned solves that run in one launch (csrc/km_persist.hip),
against the direct solution, at the edges of its tile shapes.

Tolerance: a solve ends with ||b - A x|| < eps ||b||, so its error is at most
eps ||A^-1|| ||b||; with x* the direct solution that is eps cond(A) ||x*||
at most.  With row sums of 0.01 or more and aP of at most 7, cond(A) <= 2 * 7 / 0.01
< 1e4: the bound is 1e4 eps, eps = 1e-10.
"""
import ctypes

import numpy as np
import pytest
import torch

from karman_taichi_amd import _lib
from karman_taichi_amd._lib import KmSolveInfo
from oracle import krylov

pytestmark = pytest.mark.gpu
EPS = 1e-10


def system(NX, NY, seed, diagonal):
    """A symmetric system with links of 0.5 to 1.5, an obstacle of identity
    rows where there is room, and `diagonal` added to every row."""
    rng = np.random.default_rng(seed)
    coef, b = np.zeros((5, NX, NY)), np.zeros((NX, NY))
    coef[2, 1:NX - 2, 1:NY - 1] = -(rng.random((NX - 3, NY - 2)) + 0.5)
    coef[3, 1:NX - 1, 1:NY - 2] = -(rng.random((NX - 2, NY - 3)) + 0.5)
    solid = np.zeros((NX, NY), bool)
    if NX > 12 and NY > 12:
        solid[5:8, 6:9] = True
    coef[2, :-1][solid[:-1] | solid[1:]] = 0.0
    coef[3, :, :-1][solid[:, :-1] | solid[:, 1:]] = 0.0
    coef[1, 1:], coef[4, :, 1:] = coef[2, :-1], coef[3, :, :-1]
    coef[0, 1:-1, 1:-1] = diagonal - coef[1:, 1:-1, 1:-1].sum(axis=0)
    coef[0][solid] = 1.0
    b[1:-1, 1:-1] = rng.standard_normal((NX - 2, NY - 2))
    b[solid] = 0.0
    return coef, b


def solve(dev, coef, b, flags):
    c, bt = torch.tensor(coef, device=dev), torch.tensor(b, device=dev)
    x = torch.full_like(bt, 7.0)     # every cell is written, boundary cells too
    info = KmSolveInfo()
    ctx = _lib.Context(torch.cuda.current_device(), torch.cuda.current_stream(dev).cuda_stream)
    try:
        ctx.call("km_fbicgstab", b.shape[0], b.shape[1], ctypes.c_void_p(c.data_ptr()), ctypes.c_void_p(bt.data_ptr()),
                 ctypes.c_void_p(x.data_ptr()), EPS, 0, flags, None, ctypes.byref(info))
        torch.cuda.synchronize()
    finally:
        ctx.close()
    return x.cpu().numpy(), info


def check(x, info, coef, b):
    xd = krylov.direct_solve(coef, b)
    err = np.linalg.norm(x - xd) / np.linalg.norm(xd)
    print(f"{b.shape}: {info.iterations} it, true residual {info.rel_resid_true:.1e}, error {err:.1e}")
    assert info.status == _lib.KM_OK and info.fallback == 0
    assert info.rel_resid_true < EPS
    assert err <= 1e4 * EPS


# one cell over and under the tiles (16 x 16, 16 x 32, 32 x 32, 40 x 32, 48 x 32,
# 48 x 48, 64 x 56 cells), a single tile, 256 tiles of a shape (where the next
# begins), systems of the two largest shapes, and the longest side and one past it
# (by launches)
SHAPES = [(6, 5), (18, 18), (19, 17), (50, 34), (49, 67), (258, 258), (259, 258), (258, 515), (514, 516), (602, 702),
          (802, 802), (1302, 34), (1304, 35)]


@pytest.mark.parametrize("NX,NY", SHAPES)
@pytest.mark.parametrize("mixed", [0, _lib.KM_FLAG_MIXED])
@pytest.mark.parametrize("kind", [_lib.KM_FLAG_COARSE | _lib.KM_FLAG_SYMMETRIC, _lib.KM_FLAG_SMOOTH])
def test_one_launch_matches_direct_solution(NX, NY, mixed, kind, dev):
    coef, b = system(NX, NY, NX + NY, 1.0 if kind == _lib.KM_FLAG_SMOOTH else 0.01)
    x, info = solve(dev, coef, b, kind | mixed)
    check(x, info, coef, b)


def test_coupled_boundary_rows_take_the_launches(dev):
    """A system whose boundary rows are not empty is not the one-launch
    kernel's: it says so and the solve by launches follows."""
    coef, b = system(40, 36, 3, 1.0)
    coef[0, 0, 5], b[0, 5] = 2.0, 1.0
    x, info = solve(dev, coef, b, _lib.KM_FLAG_SMOOTH)
    check(x, info, coef, b)


# one tile of 16 x 16 and of 32 x 32 (a single workgroup), one cell more,
# remainders, and 256 tiles of the first shape and one cell more
PLAIN = [(5, 4), (18, 18), (19, 18), (34, 34), (35, 34), (50, 71), (258, 258), (259, 260)]


@pytest.mark.parametrize("NX,NY", PLAIN)
@pytest.mark.parametrize("entry", ["km_bicgstab", "km_cg", "km_bicgstab_noalloc", "from_x"])
def test_plain_one_launch_matches_direct_solution(NX, NY, entry, dev):
    """The plain solves stop on the recursive residual, so the true one may
    end a little above eps: ten times, as in the parity tests."""
    coef, b = system(NX, NY, NX * NY, 0.01)
    c, bt = torch.tensor(coef, device=dev), torch.tensor(b, device=dev)
    x = torch.full_like(bt, 7.0)
    flags = 0
    if entry == "from_x":
        entry, flags = "km_bicgstab", _lib.KM_FLAG_X0 | _lib.KM_FLAG_TRUE
        x[:] = 0.0
        x[1:-1, 1:-1] = torch.tensor(np.random.default_rng(1).standard_normal((NX - 2, NY - 2)), device=dev)
    info = KmSolveInfo()
    ctx = _lib.Context(torch.cuda.current_device(), torch.cuda.current_stream(dev).cuda_stream)
    try:
        ctx.call(entry, NX, NY, ctypes.c_void_p(c.data_ptr()), ctypes.c_void_p(bt.data_ptr()),
                 ctypes.c_void_p(x.data_ptr()), EPS, 0, flags, ctypes.byref(info))
        torch.cuda.synchronize()
    finally:
        ctx.close()
    xd = krylov.direct_solve(coef, b)
    err = np.linalg.norm(x.cpu().numpy() - xd) / np.linalg.norm(xd)
    print(f"{entry} {b.shape}: {info.iterations} it, true residual {info.rel_resid_true:.1e}, error {err:.1e}")
    assert info.status == _lib.KM_OK
    assert info.rel_resid_true < 10 * EPS
    assert err <= 1e5 * EPS


@pytest.mark.parametrize("entry", ["km_bicgstab", "km_bicgstab_noalloc"])
@pytest.mark.parametrize("launches", [False, True])
def test_true_residual_decides_the_status(entry, launches, dev):
    """KM_FLAG_TRUE from a start far off: x0 of 1e7 leaves a true residual that
    the recursive one has drifted from, so restarts follow.  Wherever max_iter
    cuts them, a true residual below eps is KM_OK."""
    NX, NY = 50, 71
    coef, b = system(NX, NY, 5, 0.01)
    c, bt = torch.tensor(coef, device=dev), torch.tensor(b, device=dev)
    x0 = torch.zeros_like(bt)
    x0[1:-1, 1:-1] = 1e7 * torch.tensor(np.random.default_rng(1).standard_normal((NX - 2, NY - 2)), device=dev)
    ctx = _lib.Context(torch.cuda.current_device(), torch.cuda.current_stream(dev).cuda_stream)

    def run(max_iter):
        x, info = x0.clone(), KmSolveInfo()
        ctx.call(entry, NX, NY, ctypes.c_void_p(c.data_ptr()), ctypes.c_void_p(bt.data_ptr()),
                 ctypes.c_void_p(x.data_ptr()), EPS, max_iter, _lib.KM_FLAG_X0 | _lib.KM_FLAG_TRUE, ctypes.byref(info))
        torch.cuda.synchronize()
        return info

    try:
        if launches:
            ctx.call("km_set_tile", NX, NY, 0, 8, 32)
        whole = run(0)
        print(f"{whole.iterations} it, {whole.refinements} restarts, true residual {whole.rel_resid_true:.1e}")
        assert whole.status == _lib.KM_OK and whole.rel_resid_true < EPS and whole.refinements >= 1
        for cap in range(whole.iterations, whole.iterations // 2, -1):
            info = run(cap)
            print(f"  cap {cap}: {info.iterations} it, {info.refinements} restarts, status {info.status}, "
                  f"{info.rel_resid_true:.2e}")
            assert info.status == _lib.KM_OK or info.rel_resid_true >= EPS, cap
    finally:
        ctx.close()
