"""The binned scatter's workspace plan (host arithmetic, no kernel runs): a size that nect_grid_binned_workspace returns is
one that it, and the launches of both forms of the grid, accept."""
import ctypes
import random

import pytest
import torch

from nect_amd import _lib
from nect_amd.grid import GridDesc


def cases():
    rng = random.Random(5)
    yield GridDesc(3, 19, 4, 21, 8, 1.26), 304352, 16 << 20
    yield GridDesc(4, 16, 2, 15, 5, 1.5), 1 << 15, 1 << 30
    for _ in range(400):
        D, F, L, base = rng.choice([3, 4]), rng.choice([2, 4]), rng.randint(1, 32), rng.randint(2, 32)
        finest = 2 ** (5 + 13 * rng.random())
        grid = GridDesc(D, L, F, rng.randint(8, 22), base, max(1.0, (finest / base) ** (1 / max(1, L - 1))))
        yield grid, int(2 ** (5 + 16 * rng.random())), int(2 ** (18 + 16 * rng.random()))


def test_a_returned_size_is_accepted():
    lib = _lib.lib()
    some = 0
    for grid, slots, limit in cases():
        need = lib.nect_grid_binned_workspace(grid.struct_ref(), slots, limit)
        assert 0 <= need <= limit
        if need:
            some += 1
            again = lib.nect_grid_binned_workspace(grid.struct_ref(), slots, need)
            assert again == need, (grid.n_dims, grid.n_levels, slots, limit, need, again)
    assert some > 200


@pytest.mark.skipif(torch.cuda.is_available(), reason="hands the entry points host addresses: only where nothing can run")
def test_launches_accept_a_returned_size():
    """Without a device a launch fails; it has to get that far (the plan is checked before)."""
    lib = _lib.lib()
    at = ctypes.c_void_p(1 << 20)
    for grid, slots, limit in cases():
        slots = (slots + 31) // 32 * 32
        need = lib.nect_grid_binned_workspace(grid.struct_ref(), slots, limit)
        if not need:
            continue
        D, LF = grid.n_dims, grid.n_output_dims
        told = []
        for cols in ([0, 1, 2, 3][:D], [0, 1, 3] if D == 3 else [3, 0, 1, 2]):
            told.append(lib.nect_grid_backward_binned_rays(
                grid.struct_ref(), (ctypes.c_int32 * D)(*cols), at, at, at, at, slots // 32, 0.5, _lib.F32, at, LF, None, at,
                at, need, None))
            assert told[-1] != 0 and b"workspace" not in lib.nect_last_error(), (D, slots, limit, lib.nect_last_error())
        assert lib.nect_grid_backward_binned(grid.struct_ref(), at, slots, D, _lib.F32, at, LF, None, at, at, need, None) != 0
        assert b"workspace" not in lib.nect_last_error(), (D, slots, limit, lib.nect_last_error())


def test_sizes_are_kept_per_level_table():
    """Two grids of the same dimensions, parameter count and base resolution, one with a hashed level where the other's is
    dense (lists of another capacity): each gets its own size."""
    from nect_amd.fused import BinnedScatter

    dense, hashed = GridDesc(3, 2, 4, 12, 16, 1.0), GridDesc(3, 2, 4, 12, 16, 2.0)
    assert dense.n_params == hashed.n_params
    slots = 1 << 22
    own = [BinnedScatter("cpu", 12 << 30)._need([g], slots) for g in (dense, hashed)]
    assert own[0] > own[1] > 0
    for order in ((dense, hashed), (hashed, dense)):
        kept = BinnedScatter("cpu", 12 << 30)
        assert {g: kept._need([g], slots) for g in order} == dict(zip((dense, hashed), own))


# (grid, samples, whether the records' schedule was the faster one by more than 5 % either way: the measured steps that
# BinnedScatter.least lists, and a dynamic preset's training batches)
@pytest.mark.parametrize("args,slots,binned", [
    ((3, 16, 2, 19, 16, 1.5), 1 << 14, False), ((3, 16, 2, 19, 16, 1.5), 1 << 15, True),
    ((3, 16, 2, 21, 16, 1.5), 1 << 15, False), ((3, 16, 2, 21, 16, 1.5), 1 << 16, True),
    ((3, 16, 2, 23, 16, 1.5), 1 << 17, False), ((3, 19, 4, 21, 8, 1.26), 1 << 17, True),
    ((3, 19, 4, 22, 8, 1.26), 1 << 16, False), ((3, 19, 4, 23, 8, 1.26), 1 << 19, False),
    ((3, 19, 4, 23, 8, 1.26), 1 << 20, True), ((4, 16, 2, 20, 16, 1.5), 1 << 15, True),
    ((3, 23, 4, 23, 16, 1.17), 1_000_000, False), ((3, 23, 4, 23, 16, 1.17), 2_499_840, True)])
def test_batches_take_the_faster_schedule(args, slots, binned):
    from nect_amd.fused import BinnedScatter

    assert (slots >= BinnedScatter.least(GridDesc(*args))) == binned
