"""Which path a solve takes, by the context's counts of one-launch solves, and
the way back from a launch that gives up.

Solutions against the direct one.  Tolerances as in test_gpu_one_launch.py: the
error is at most cond(A) < 1e4 times the true residual, eps = 1e-10, and the
plain solves, which stop on the recursive residual, may end at ten times eps.
"""
import ctypes
import functools

import numpy as np
import pytest
import torch

from karman_taichi_amd import _lib
from karman_taichi_amd._lib import KmSolveInfo, ptr
from oracle import krylov
from test_gpu_one_launch import EPS, SHAPES, system

pytestmark = pytest.mark.gpu

COARSE = _lib.KM_FLAG_COARSE | _lib.KM_FLAG_SYMMETRIC


class Solver:
    """One context; solve() by any entry, counts() of its one-launch solves."""

    def __init__(self, dev):
        self.dev = dev
        self.ctx = _lib.Context(torch.cuda.current_device(), torch.cuda.current_stream(dev).cuda_stream)

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        self.ctx.close()

    def counts(self):
        return self.ctx.one_launch_counts()

    def solve(self, entry, coef, b):
        NX, NY = b.shape
        c, bt = torch.tensor(coef, device=self.dev), torch.tensor(b, device=self.dev)
        x, info = torch.full_like(bt, 7.0), KmSolveInfo()
        if entry == "from_x":
            x[:] = 0.0
            x[1:-1, 1:-1] = torch.tensor(np.random.default_rng(1).standard_normal((NX - 2, NY - 2)), device=self.dev)
        flags = {"from_x": _lib.KM_FLAG_X0 | _lib.KM_FLAG_TRUE, "coarse": COARSE, "smooth": _lib.KM_FLAG_SMOOTH,
                 "coarse_mixed": COARSE | _lib.KM_FLAG_MIXED, "smooth_mixed": _lib.KM_FLAG_SMOOTH | _lib.KM_FLAG_MIXED,
                 "pair": _lib.KM_FLAG_SMOOTH, "group": COARSE}.get(entry, 0)
        if entry == "pair":
            y, info2 = torch.full_like(bt, 7.0), KmSolveInfo()
            self.ctx.call("km_fbicgstab2", NX, NY, ptr(c), ptr(bt), ptr(x), NX, NY, ptr(c), ptr(bt), ptr(y), EPS, 0,
                          flags, ctypes.byref(info), ctypes.byref(info2))
            torch.cuda.synchronize()
            assert torch.equal(x, y) and info2.status == info.status
        elif entry == "group":
            sizes = [(ctypes.c_int * 1)(v) for v in (NX, NY)]
            ptrs = [(ctypes.c_void_p * 1)(t.data_ptr()) for t in (c, bt, x)]
            self.ctx.call("km_fbicgstab_n", 1, *sizes, *ptrs, EPS, 0, flags, ctypes.byref(info))
        elif flags and entry != "from_x":
            self.ctx.call("km_fbicgstab", NX, NY, ptr(c), ptr(bt), ptr(x), EPS, 0, flags, None, ctypes.byref(info))
        else:
            self.ctx.call("km_bicgstab" if entry == "from_x" else entry, NX, NY, ptr(c), ptr(bt), ptr(x), EPS, 0,
                          flags, ctypes.byref(info))
        torch.cuda.synchronize()
        xd = direct(coef.tobytes(), b.tobytes(), b.shape)
        err = np.linalg.norm(x.cpu().numpy() - xd) / np.linalg.norm(xd)
        print(f"{entry} {b.shape}: {info.iterations} it, true residual {info.rel_resid_true:.1e}, error {err:.1e}, "
              f"one launch {self.counts()}")
        assert info.status == _lib.KM_OK and info.fallback == 0
        plain = entry.startswith("km_") or entry == "from_x"
        assert info.rel_resid_true < (10 * EPS if plain else EPS)
        assert err <= (1e5 * EPS if plain else 1e4 * EPS)


@functools.lru_cache(maxsize=4)
def direct(coef, b, shape):
    return krylov.direct_solve(np.frombuffer(coef).reshape((5,) + shape), np.frombuffer(b).reshape(shape))


@pytest.mark.parametrize("entry", ["coarse", "coarse_mixed", "smooth", "smooth_mixed"])
def test_preconditioned_sizes_take_one_launch(entry, dev):
    """Every size of the one-launch tests but the side of 1302 cells."""
    for NX, NY in SHAPES:
        coef, b = system(NX, NY, NX + NY, 1.0 if entry.startswith("smooth") else 0.01)
        c, bt = torch.tensor(coef, device=dev), torch.tensor(b, device=dev)
        x, info = torch.zeros_like(bt), KmSolveInfo()
        flags = (_lib.KM_FLAG_SMOOTH if entry.startswith("smooth") else COARSE)
        flags |= _lib.KM_FLAG_MIXED if entry.endswith("mixed") else 0
        with Solver(dev) as s:
            s.ctx.call("km_fbicgstab", NX, NY, ptr(c), ptr(bt), ptr(x), EPS, 0, flags, None, ctypes.byref(info))
            run, refused, gave_up = s.counts()
        assert refused == gave_up == 0, (NX, NY)
        assert (run > 0) == (max(NX, NY) - 2 <= 1300), (NX, NY)


# the plain kernel's five shapes: 16 x 16 and 32 x 32 alone, 16 x 16, 32 x 32,
# 40 x 32, 48 x 48 and 64 x 64 cells (1024 threads), with remainders; and a
# system of more tiles than compute units, by launches
PLAIN = [(18, 17, 1), (34, 33, 1), (51, 40, 1), (260, 270, 1), (516, 515, 1), (645, 525, 1), (6148, 52, 1)]


@pytest.mark.parametrize("NX,NY,run", PLAIN + [(16400, 36, 0)])
@pytest.mark.parametrize("entry", ["km_bicgstab", "km_cg", "km_bicgstab_noalloc", "from_x"])
def test_plain_shapes_take_one_launch(NX, NY, run, entry, dev):
    if entry == "km_bicgstab_noalloc" and NX * NY > _lib.NOALLOC_MAX_CELLS:
        pytest.skip("larger than the library's scratch array")
    coef, b = system(NX, NY, NX * NY, 0.01)
    with Solver(dev) as s:
        s.solve(entry, coef, b)
        counts = s.counts()
        assert counts[1:] == (0, 0)
        assert (counts[0] > 0) == bool(run)


ENTRIES = ["km_bicgstab", "km_cg", "km_bicgstab_noalloc", "from_x", "coarse", "coarse_mixed", "smooth",
           "smooth_mixed", "pair", "group"]


@pytest.mark.parametrize("entry", ENTRIES)
def test_a_launch_that_gives_up_is_solved_by_launches(entry, dev):
    """The launch leaves at its first exchange and the same call solves by
    launches; the next solve is one launch again; after two that gave up the
    context stays with the launches."""
    coef, b = system(100, 71, 9, 0.5)
    with Solver(dev) as s:
        s.ctx.call("km_one_launch_give_up", 1)
        s.solve(entry, coef, b)
        first = s.counts()
        assert first[1:] == (0, 1)
        s.solve(entry, coef, b)
        again = s.counts()
        assert again[0] > first[0] and again[1:] == (0, 1)
        s.ctx.call("km_one_launch_give_up", 1)
        s.solve(entry, coef, b)
        closed = s.counts()
        assert closed[1:] == (0, 2)
        s.solve(entry, coef, b)
        assert s.counts() == closed


def test_give_ups_of_all_entries_count_together(dev):
    coef, b = system(100, 71, 9, 0.5)
    with Solver(dev) as s:
        s.ctx.call("km_one_launch_give_up", 2)
        s.solve("km_bicgstab_noalloc", coef, b)
        s.solve("smooth", coef, b)
        for entry in ENTRIES:
            s.solve(entry, coef, b)
        assert s.counts() == (0, 0, 2)


def with_rim(coef, b):
    """The same system with a coupled identity row on the rim."""
    coef, b = coef.copy(), b.copy()
    coef[0, 0, 5], b[0, 5] = 2.0, 1.0
    return coef, b


@pytest.mark.parametrize("entry", ENTRIES)
def test_a_refused_size_rests(entry, dev):
    """A program whose systems have identity rows on the rim pays for one
    refusal in 32 solves, and every system is solved whichever path it takes."""
    coef, b = system(100, 71, 9, 0.5)
    with Solver(dev) as s:
        s.solve(entry, *with_rim(coef, b))
        first = s.counts()
        assert first[0] == first[2] == 0 and first[1] in (1, 2)
        for _ in range(3):
            s.solve(entry, *with_rim(coef, b))
            s.solve(entry, coef, b)
        assert s.counts() == first
        s.solve(entry, *system(90, 71, 9, 0.5))          # another size does not rest
        assert s.counts()[0] > 0 and s.counts()[1] == first[1]
        run = s.counts()[0]
        for _ in range(40):
            s.solve(entry, coef, b)
        assert s.counts()[0] > run and s.counts()[1] == first[1]
