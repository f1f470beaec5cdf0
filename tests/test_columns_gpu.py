"""The encoder over detector columns (nect_ray_order_columns, nect_grid_encode_ray_columns): the order is a permutation
by column, 64-row patch and row; the features are bit for bit those of nect_grid_encode_rays (tested against the oracle)."""
import numpy as np
import pytest
import torch

from tests.helpers import cfg1_geometry, product_struct, seeded_batch

pytestmark = pytest.mark.gpu


# levels x features whose samples are 4 to 256 bytes: one 16-byte piece, odd counts, few samples staged at a time
@pytest.mark.parametrize("args", [(3, 16, 2, 14, 8, 1.5), (3, 3, 2, 9, 6, 1.6), (3, 5, 4, 13, 6, 1.9), (3, 24, 4, 12, 5, 1.2),
                                  (3, 1, 2, 9, 4, 1.0), (4, 16, 2, 14, 5, 1.4), (4, 7, 4, 12, 4, 1.6), (4, 8, 4, 13, 4, 1.5)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,S,order", [(1, 1, False), (33, 32, True), (700, 61, False), (2049, 40, True)])
def test_encode_matches(device, args, dtype, B, S, order):
    """Rows (packed, and padded by a level's features) and planes; odd numbers of rays and samples, rays that miss the
    volume (no tile) and tiles that end early; slots of no tile stay as they were."""
    from nect_amd import _lib
    from nect_amd.grid import GridDesc
    from nect_amd.sampling import ct_sampling as cs

    print(f"[columns] encode {args} {dtype} B={B} S={S} order={order}", flush=True)
    desc = GridDesc(*args)
    F, LF = desc.n_features, desc.n_output_dims
    geo = cfg1_geometry()
    g = product_struct(geo.c_struct_fields())
    idx, jit, off = seeded_batch(64 * 64, B, seed=B, det_offset_scale=1.0)
    ridx = torch.from_numpy(idx[:B]).to(device)
    if B > 100:
        ridx[::13] = 64 * 64 + 5     # not a pixel: an empty ray
    if order:
        ridx = ridx[column_order(g, ridx, B, 0, device).long()].contiguous()
    rays = cs.ray_setup(ridx, g, 0.4, S, B, 0, geo.max_distance_traveled / S, True, torch.from_numpy(jit).to(device),
                        torch.from_numpy(off).to(device))
    mt = cs.tiles_needed(B, S)
    tile_offsets, tile_ray, n_tiles = cs.ray_tiles(rays, mt)
    gen = torch.Generator(device=device).manual_seed(S)
    table = torch.randn(desc.n_params, device=device, generator=gen).to(dtype)
    st = _lib.stream_of(device)
    for grouped, stride in [(0, LF), (0, LF + F)] + ([(1, LF)] if desc.n_levels % 8 == 0 else []):
        out = []
        for name in ("nect_grid_encode_rays", "nect_grid_encode_ray_columns"):
            o = torch.full((mt * 32 * stride,), 7.0, device=device, dtype=dtype)
            if name == "nect_grid_encode_rays":
                _lib.call(name, desc.struct_ref(), _lib.dtype_code(dtype), table.data_ptr(), _lib.ptr(rays),
                          _lib.ptr(tile_offsets), _lib.ptr(tile_ray), _lib.ptr(n_tiles), mt, 0.3, o.data_ptr(), stride,
                          grouped, st)
            else:
                _lib.call(name, desc.struct_ref(), _lib.dtype_code(dtype), table.data_ptr(), _lib.ptr(rays),
                          _lib.ptr(tile_offsets), B, S, mt, 0.3, o.data_ptr(), stride, grouped, st)
            torch.cuda.synchronize()
            out.append(o)
        used = int(n_tiles.item()) * 32
        if grouped:
            a, b = (o.view(8, mt * 32, LF // 8)[:, :used] for o in out)
            rest = out[1].view(8, mt * 32, LF // 8)[:, used:]
        else:
            a, b = (o.view(mt * 32, stride)[:used, :LF] for o in out)
            rest = torch.cat([out[1].view(mt * 32, stride)[used:].flatten(), out[1].view(mt * 32, stride)[:, LF:].flatten()])
        assert torch.equal(a, b), (grouped, stride)
        assert bool((rest == 7.0).all())


def column_order(geo, ridx, num, start, device):
    from nect_amd import _lib

    need = int(_lib.lib().nect_ray_order_columns_workspace(geo._struct()))
    ws = torch.empty(need, dtype=torch.uint8, device=device)
    order = torch.full((num,), -1, dtype=torch.int32, device=device)
    _lib.call("nect_ray_order_columns", geo._struct(), _lib.ptr(ridx), ridx.numel(), num, start, _lib.ptr(order),
              _lib.ptr(ws), ws.numel(), _lib.stream_of(device))
    torch.cuda.synchronize()
    return order


@pytest.mark.parametrize("rows,cols,unique", [(64, 64, False), (200, 37, True), (1, 300, True), (130, 3, False)])
def test_order(device, rows, cols, unique):
    """Repeated pixels, pixels outside the detector and slots past the end of the index; a column's patches of 64 rows
    follow one another, distinct pixels of a patch from the first row to the last, rays without a pixel last."""
    from oracle.geometry import OracleGeometry

    print(f"[columns] order {rows}x{cols} unique={unique}", flush=True)
    geo = product_struct(OracleGeometry(mode="cone", nDetector=(rows, cols), dDetector=(1.0, 1.0), DSD=1000.0, DSO=500.0,
                                        nVoxel=(64, 64, 64), dVoxel=(0.5, 0.5, 0.5)).c_struct_fields())
    rng = np.random.default_rng(rows)
    n_pix, start = rows * cols, 10
    idx = (rng.permutation(np.arange(-40, n_pix + 40)) if unique else rng.integers(-50, n_pix + 50, size=3000)).astype(np.int64)
    num = idx.size
    o = column_order(geo, torch.from_numpy(idx).to(device), num, start, device).cpu().numpy()
    assert np.array_equal(np.sort(o), np.arange(num))
    pix = np.array([idx[start + t] if start + t < idx.size else -1 for t in o])
    valid = (pix >= 0) & (pix < n_pix)
    row, col = np.where(valid, pix // cols, 0), np.where(valid, pix % cols, 0)
    per = (rows + 63) // 64
    patch = np.where(valid, col * per + row // 64, per * cols)
    assert np.all(np.diff(patch) >= 0)
    for p in np.unique(patch[valid]):
        sel = patch == p
        if len(np.unique(pix[sel])) == sel.sum():
            assert np.all(np.diff(row[sel]) > 0), p


@pytest.mark.parametrize("B,S,order", [(33, 32, True), (700, 61, False)])
def test_encode_widest_float32(device, B, S, order):
    """32 levels of 4 float32 features: one sample of 512 bytes staged at a time takes more than 64 KiB of LDS."""
    test_encode_matches(device, (3, 32, 4, 11, 4, 1.15), torch.float32, B, S, order)
