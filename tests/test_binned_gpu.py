"""The binned table gradient (nect_grid_backward_binned, nect_grid_backward_binned_rays) against a float64 sum of the
same contributions, formed from nect_grid_index's corners and weights (bit-exact against the oracle).

Tolerance per entry: (32 + c) 2^-24 times the sum of the absolute contributions, c the entry's number of contributions:
each contribution is a product of at most six float32 factors and a float32 sum over at most 16 lanes twice (under 32
roundings); those added straight to the gradient (a full list, a pair across two bins) add one rounding each.  Onto a
gradient that is not zero, a chunk adds an entry's sum in at most 64 parts, each rounding to 2^-24 of the running value:
min(c, 64 chunks) + 1 such roundings of the starting value."""
import ctypes

import numpy as np
import pytest
import torch

from tests.helpers import cfg1_geometry, product_struct, seeded_batch

pytestmark = pytest.mark.gpu


def reference(desc, x, dout):
    """(gradient, tolerance, contributions) float64 [n_params] for positions x [n, D] and dout [n, L*F] float64."""
    from nect_amd import grid as ng

    idx, w = ng.index(desc, x.contiguous())
    L, F = desc.n_levels, desc.n_features
    off = torch.tensor(desc.offset[:L], device=x.device, dtype=torch.int64)
    ent = (idx.long() & 0xFFFFFFFF) + off[None, :, None]
    v = w.double()[..., None] * dout.view(-1, L, 1, F)
    flat = (ent[..., None] * F + torch.arange(F, device=x.device)).flatten()
    ref = torch.zeros(desc.n_params, dtype=torch.float64, device=x.device)
    mag, cnt = torch.zeros_like(ref), torch.zeros_like(ref)
    ref.index_add_(0, flat, v.flatten())
    mag.index_add_(0, flat, v.abs().flatten())
    cnt.index_add_(0, flat, torch.ones_like(flat, dtype=torch.float64))
    return ref, (32 + cnt) * 2.0 ** -24 * mag, cnt


def workspace(desc, slots, max_bytes, device):
    from nect_amd import _lib

    need = int(_lib.lib().nect_grid_binned_workspace(desc.struct_ref(), slots, max_bytes))
    assert 0 < need <= max_bytes
    return torch.empty(need, dtype=torch.uint8, device=device)


def check(out, start, want, chunks=8):
    ref, tol, cnt = want
    tol = tol + (cnt.clamp(max=64 * chunks) + 1) * 2.0 ** -24 * start.double().abs() + 1e-30
    err = (out.double() - start.double() - ref).abs()
    assert bool((err <= tol).all()), float((err - tol).max())


# tables: one bin (512 entries), several bins dense and hashed, a level that just fills a bin, growth with many levels
GRIDS = [(3, 3, 2, 9, 6, 1.6), (3, 16, 2, 14, 8, 1.5), (3, 5, 4, 15, 16, 1.9), (4, 4, 2, 15, 5, 1.7), (4, 3, 4, 13, 4, 2.0),
         (3, 32, 2, 12, 4, 1.2), (3, 2, 2, 12, 16, 1.0)]


@pytest.mark.parametrize("args", GRIDS)
@pytest.mark.parametrize("n,dtype,pad,crowd", [(1, torch.float32, 0, False), (31, torch.float16, 2, False),
                                               (513, torch.float32, 4, False), (20011, torch.bfloat16, 8, False),
                                               (70001, torch.float32, 1, False), (30000, torch.float16, 0, True)])
def test_points(device, args, n, dtype, pad, crowd):
    """Random points (crowd: all within one cell of the finest level, so that a bin's list overflows), dout rows of
    several types, strides and alignments, a tenth of them zero, added onto a gradient that is not zero; one chunk and
    several."""
    from nect_amd import _lib
    from nect_amd.grid import GridDesc

    print(f"[binned] points {args} n={n} {dtype} pad={pad} crowd={crowd}", flush=True)
    desc = GridDesc(*args)
    D, LF = desc.n_dims, desc.n_output_dims
    g = torch.Generator(device=device).manual_seed(n)
    x = torch.rand((n, D + 1), device=device, generator=g)
    if crowd:
        x = 0.4 + x * 1e-4
    x[:: 17] = 1.0
    d = torch.randn((n, LF + pad), device=device, generator=g).to(dtype)
    d[::10] = 0
    scale = None if dtype == torch.float32 else torch.full((1,), 0.125, device=device)
    want = reference(desc, x[:, :D], d[:, :LF].double() * (1.0 if scale is None else 0.125))
    start = torch.randn(desc.n_params, device=device, generator=g) * 1e-3
    whole = workspace(desc, n, 1 << 32, device)
    for ws in [whole] + ([workspace(desc, n, whole.numel() // 3 + 65536, device)] if n > 20000 else []):
        out = start.clone()
        _lib.call("nect_grid_backward_binned", desc.struct_ref(), x.data_ptr(), n, D + 1, _lib.dtype_code(dtype),
                  d.data_ptr(), LF + pad, _lib.ptr(scale), out.data_ptr(), ws.data_ptr(), ws.numel(),
                  _lib.stream_of(device))
        torch.cuda.synchronize()
        check(out, start, want)


@pytest.mark.parametrize("args", [(3, 4, 2, 17, 24, 1.7), (3, 3, 4, 16, 30, 1.5), (4, 3, 2, 16, 9, 2.0)])
def test_crowded_points(device, args):
    """So many points in a few cells that the bins' lists overflow and the rest goes straight to the gradient."""
    from nect_amd import _lib
    from nect_amd.grid import GridDesc

    print(f"[binned] crowded points {args}", flush=True)
    desc = GridDesc(*args)
    n, D, LF = 400003, desc.n_dims, desc.n_output_dims
    g = torch.Generator(device=device).manual_seed(7)
    x = 0.3 + torch.rand((n, D), device=device, generator=g) * 0.02
    d = torch.randn((n, LF), device=device, generator=g)
    want = reference(desc, x, d.double())
    ws = workspace(desc, n, 1 << 30, device)
    out = torch.zeros(desc.n_params, device=device)
    _lib.call("nect_grid_backward_binned", desc.struct_ref(), x.data_ptr(), n, D, _lib.F32, d.data_ptr(), LF, None,
              out.data_ptr(), ws.data_ptr(), ws.numel(), _lib.stream_of(device))
    torch.cuda.synchronize()
    check(out, torch.zeros_like(out), want)


@pytest.mark.parametrize("args", GRIDS)
@pytest.mark.parametrize("cols", [None, "t last", "t first", "no t"])
@pytest.mark.parametrize("B,S,t", [(3, 7, 0.0), (700, 64, 0.37), (4096, 40, 1.0)])
def test_rays(device, args, cols, B, S, t):
    """Samples of cone-beam rays, with the time as the last dimension (folded), as another one and not at all."""
    from nect_amd import _lib
    from nect_amd.grid import GridDesc
    from nect_amd.sampling import ct_sampling as cs

    desc = GridDesc(*args)
    D, LF = desc.n_dims, desc.n_output_dims
    pick = {None: (0, 1, 2, 3)[:D], "t last": (1, 0, 2, 3)[:D] if D == 4 else (2, 0, 3),
            "t first": (3, 1, 0, 2)[:D], "no t": (2, 1, 0, 0)[:D]}[cols]
    print(f"[binned] rays {args} cols={pick} B={B} S={S} t={t}", flush=True)
    geo = cfg1_geometry()
    idx, jit, off = seeded_batch(64 * 64, B, seed=B)
    rays = cs.ray_setup(torch.from_numpy(idx[:B]).to(device), product_struct(geo.c_struct_fields()), 0.4, S, B, 0,
                        geo.max_distance_traveled / S, True, torch.from_numpy(jit).to(device),
                        torch.from_numpy(off).to(device))
    mt = cs.tiles_needed(B, S)
    tile_offsets, tile_ray, n_tiles = cs.ray_tiles(rays, mt)
    pos, valid = cs.ray_positions(rays, tile_offsets, tile_ray, n_tiles, mt)
    zyxt = torch.cat([pos, torch.full_like(pos[:, :1], t)], dim=1)
    g = torch.Generator(device=device).manual_seed(S)
    d = torch.randn((mt * 32, LF), device=device, generator=g)
    live = valid != 0
    want = reference(desc, zyxt[live][:, list(pick)], d[live].double())
    start = torch.zeros(desc.n_params, device=device)
    ws = workspace(desc, mt * 32, 1 << 30, device)
    out = start.clone()
    _lib.call("nect_grid_backward_binned_rays", desc.struct_ref(),
              None if cols is None else (ctypes.c_int32 * D)(*pick), _lib.ptr(rays), _lib.ptr(tile_offsets),
              _lib.ptr(tile_ray), _lib.ptr(n_tiles), mt, t, _lib.F32, d.data_ptr(), LF, None, out.data_ptr(),
              ws.data_ptr(), ws.numel(), _lib.stream_of(device))
    torch.cuda.synchronize()
    check(out, start, want)


def test_refusals(device):
    """A grid whose levels need too many bins has no workspace, a short or misaligned workspace is refused, and a
    non-finite gradient reaches the table."""
    from nect_amd import _lib
    from nect_amd.grid import GridDesc

    lib = _lib.lib()
    big = GridDesc(3, 2, 4, 25, 256, 2.0)
    assert lib.nect_grid_binned_workspace(big.struct_ref(), 1 << 16, 1 << 40) == 0
    desc = GridDesc(3, 4, 2, 12, 8, 1.5)
    assert lib.nect_grid_binned_workspace(desc.struct_ref(), 1 << 16, 100) == 0
    n = 1000
    x = torch.rand((n, 3), device=device)
    d = torch.ones((n, 8), device=device)
    grad = torch.zeros(desc.n_params, device=device)
    ws = workspace(desc, n, 1 << 30, device)

    def run(p, size):
        return lib.nect_grid_backward_binned(desc.struct_ref(), x.data_ptr(), n, 3, _lib.F32, d.data_ptr(), 8, None,
                                             grad.data_ptr(), p, size, _lib.stream_of(device))

    assert run(ws.data_ptr(), 64) != 0 and b"workspace" in lib.nect_last_error()
    assert run(ws.data_ptr() + 8, ws.numel() - 8) != 0 and b"aligned" in lib.nect_last_error()
    assert not bool(grad.any())
    d[5, 3] = float("inf")
    d[6, 0] = float("nan")
    assert run(ws.data_ptr(), ws.numel()) == 0
    torch.cuda.synchronize()
    assert not bool(torch.isfinite(grad).all())
    assert np.isfinite(grad.cpu().numpy()).sum() >= grad.numel() - 64


@pytest.mark.parametrize("args", [(3, 3, 4, 19, 100, 1.6), (3, 2, 4, 21, 300, 1.5)])
@pytest.mark.parametrize("held", [None, 2, 1, 0])
def test_points_with_a_coordinate_held(device, args, held):
    """Points that all have one coordinate, on levels of 256 bins and more, whose bins interleave; in chunks, too."""
    from nect_amd import _lib
    from nect_amd.grid import GridDesc

    print(f"[binned] held coordinate {args} {held}", flush=True)
    desc = GridDesc(*args)
    n, LF = 90001, desc.n_output_dims
    g = torch.Generator(device=device).manual_seed(11)
    x = torch.rand((n, 3), device=device, generator=g)
    if held is not None:
        x[:, held] = 0.37
    d = torch.randn((n, LF), device=device, generator=g)
    want = reference(desc, x, d.double())
    whole = workspace(desc, n, 1 << 32, device)
    for ws in (whole, workspace(desc, n, whole.numel() // 3 + (1 << 20), device)):
        out = torch.zeros(desc.n_params, device=device)
        _lib.call("nect_grid_backward_binned", desc.struct_ref(), x.data_ptr(), n, 3, _lib.F32, d.data_ptr(), LF, None,
                  out.data_ptr(), ws.data_ptr(), ws.numel(), _lib.stream_of(device))
        torch.cuda.synchronize()
        check(out, torch.zeros_like(out), want)


@pytest.mark.parametrize("log2T", [19, 21])
def test_points_with_the_last_coordinate_held_are_no_slower_than_atomics(device, log2T):
    """Lists that overflow send their records to the table one by one: the records' gradient of half a million points at one
    time then took 1.1 to 1.2 times as long as the atomics'; with the records spread, half as long."""
    from nect_amd import _lib
    from nect_amd.grid import GridDesc

    print(f"[binned] held coordinate, time, T = 2^{log2T}", flush=True)
    desc = GridDesc(3, 23, 4, log2T, 16, 1.17)
    n, LF = 1 << 19, desc.n_output_dims
    g = torch.Generator(device=device).manual_seed(12)
    x = torch.rand((n, 3), device=device, generator=g)
    x[:, 2] = 0.37
    d = torch.randn((n, LF), device=device, generator=g)
    out = torch.zeros(desc.n_params, device=device)
    ws = workspace(desc, n, 2 << 30, device)
    st = _lib.stream_of(device)

    def binned():
        _lib.call("nect_grid_backward_binned", desc.struct_ref(), x.data_ptr(), n, 3, _lib.F32, d.data_ptr(), LF, None,
                  out.data_ptr(), ws.data_ptr(), ws.numel(), st)

    def atomics():
        _lib.call("nect_grid_backward", desc.struct_ref(), x.data_ptr(), n, 3, d.data_ptr(), LF, out.data_ptr(), st)

    best = {}
    for f in (binned, atomics, binned, atomics, binned, atomics):
        f()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(4):
            f()
        e1.record()
        torch.cuda.synchronize()
        best[f] = min(best.get(f, 1e9), e0.elapsed_time(e1))
    print(f"[binned] {best[binned] / 4:.3f} ms, atomics {best[atomics] / 4:.3f}", flush=True)
    assert best[binned] < best[atomics]
