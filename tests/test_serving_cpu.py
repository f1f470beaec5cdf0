"""Host logic of the export server: the brick traversal's codes and lengths, and that positions map onto
the grid one to one (the kernel's mapping, restated in numpy)."""
import numpy as np

from nect_amd.serving import traversal


def _voxels(n, code, length):
    """(iz, iy, ix, valid) for every traversal position, as the query kernel maps them."""
    v = np.arange(length, dtype=np.int64)
    if code == 0:
        iz, r = np.divmod(v, n[1] * n[2])
        iy, ix = np.divmod(r, n[2])
        return iz, iy, ix, iz < n[0]
    lz, ly, lx = (code >> 8) & 15, (code >> 4) & 15, code & 15
    ib = lz + ly + lx
    b, inner = v >> ib, v & ((1 << ib) - 1)
    nbx, nby = -(-n[2] // (1 << lx)), -(-n[1] // (1 << ly))
    bz, r = np.divmod(b, nby * nbx)
    by, bx = np.divmod(r, nbx)
    iz = (bz << lz) + (inner >> (ly + lx))
    iy = (by << ly) + ((inner >> lx) & ((1 << ly) - 1))
    ix = (bx << lx) + (inner & ((1 << lx) - 1))
    return iz, iy, ix, (iz < n[0]) & (iy < n[1]) & (ix < n[2])


def test_traversal_codes():
    assert traversal((512, 512, 512)) == (0x222, 512 ** 3)
    assert traversal((1, 512, 512)) == (0x022, 512 ** 2)
    assert traversal((512, 512, 1)) == (0x220, 512 ** 2)
    assert traversal((7, 33, 40)) == (0x222, 8 * 36 * 40)
    assert traversal((3, 2, 1)) == (0x110, 4 * 2 * 1)
    assert traversal((1, 1, 1)) == (0, 1)
    assert traversal((64, 64, 64), bricks=False) == (0, 64 ** 3)


def test_traversal_covers_every_voxel_once():
    for n in [(7, 33, 40), (1, 512, 9), (5, 1, 3), (65, 66, 67), (4, 4, 4), (2, 3, 17)]:
        code, length = traversal(n)
        iz, iy, ix, ok = _voxels(n, code, length)
        flat = (iz[ok] * n[1] + iy[ok]) * n[2] + ix[ok]
        assert np.array_equal(np.sort(flat), np.arange(n[0] * n[1] * n[2])), n
        # a position past the traversal maps outside the grid
        iz2, iy2, ix2, ok2 = _voxels(n, code, length + 64)
        assert not ok2[length:].any()


def _stacked_voxels(n, code, length):
    """As _voxels for NECT_BRICK_STACKED: layers of bricks stacked up to 32 voxels along z, z fastest in a stack."""
    lz, ly, lx = (code >> 8) & 15, (code >> 4) & 15, code & 15
    nbz, nby, nbx = (-(-k // (1 << l)) for k, l in zip(n, (lz, ly, lx)))
    order = []
    for z0 in range(0, nbz, 32 >> lz):
        nz = min(32 >> lz, nbz - z0) << lz
        y, x, yy, xx, zz = np.meshgrid(np.arange(nby), np.arange(nbx), np.arange(1 << ly), np.arange(1 << lx),
                                       np.arange(nz), indexing="ij")
        order.append(np.stack([(z0 << lz) + zz, (y << ly) + yy, (x << lx) + xx], -1).reshape(-1, 3))
    iz, iy, ix = np.concatenate(order)[:length].T
    return iz, iy, ix, (iz < n[0]) & (iy < n[1]) & (ix < n[2])


def test_stacked_traversal_covers_every_voxel_once():
    for n in [(7, 33, 40), (1, 512, 9), (5, 1, 3), (65, 66, 67), (37, 5, 6), (4, 4, 4), (2, 3, 17)]:
        code, length = traversal(n)
        iz, iy, ix, ok = _stacked_voxels(n, code, length)
        assert iz.size == length
        flat = (iz[ok] * n[1] + iy[ok]) * n[2] + ix[ok]
        assert np.array_equal(np.sort(flat), np.arange(n[0] * n[1] * n[2])), n


def test_coarse_layers_are_not_stacked():
    """Voxels far apart along z share no cache lines there (17 slices of 512^2 took 8 to 11 % longer stacked)."""
    from nect_amd.serving import QueryRequest, slice_request, subvolume_request, volume_request

    for r in (volume_request(0.1), subvolume_request((3, 4, 5), 64, 0.1), slice_request("xy", 0.3, 0.1),
              slice_request("xz", 0.3, 0.1), QueryRequest((1, 1, 1), (0.1,) * 3, (0.1,) * 3),
              QueryRequest((128, 512, 512), (0.0,) * 3, (1.0,) * 3)):
        assert r.fine_along_z(), r.n
    for n in ((17, 512, 512), (3, 200, 200)):
        assert not QueryRequest(n, (0.1,) * 3, (0.9,) * 3).fine_along_z()
