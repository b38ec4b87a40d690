"""CPU check of the addressing of the adjoint's derivative adjoints (astaroth_amd/csrc/adjoint.hip), which have no halo
and rows padded to 64 bytes: row = nx rounded up to a line, plane = row ny, field = plane nz, NG fields. For every column
block, lane and round of transpose_block's DMA, and for every column, the byte offset within a plane

    (gx + row gy) s + 4 wd,   gx, gy wrapped into the grid, s = sizeof(real), wd the dword of a value

fits 32 bits signed and is the intended value's, and the LDS dwords written (wave base + lane) are those of the tile
cell that the stencils read there, each field-plane within its stride. The local stage writes the same layout."""
import numpy as np
import pytest

R = 3
TY = 16
GRIDS = [(3, 3, 3), (5, 4, 3), (17, 33, 70), (65, 17, 9), (72, 60, 50), (128, 48, 67), (200, 150, 100), (1024, 16, 16),
         (16, 1024, 16), (384, 384, 384)]


def tile(size, tx):
    lx, ly, wpe = tx + 2 * R, TY + 2 * R, size // 4
    nw = tx * TY // 64
    lpw = lx * ly * wpe
    nr = ((lpw + 63) // 64 + nw - 1) // nw
    return lx, ly, wpe, nw, lpw, nr, nr * nw * 64 // wpe


@pytest.mark.parametrize("size,tx", [(4, 64), (4, 32), (4, 16), (8, 32), (8, 16)])
@pytest.mark.parametrize("n", GRIDS)
def test_transpose_block_addresses(n, size, tx):
    nx, ny, nz = n
    line = 64 // size
    row = -(-nx // line) * line
    plane = row * ny
    assert row >= nx and row * size % 64 == 0
    lx, ly, wpe, nw, lpw, nr, lps = tile(size, tx)
    assert 8 * 2 * lps * size <= 160 * 1024  # two buffers of at most eight field-planes
    wave, r, lane = np.meshgrid(np.arange(nw), np.arange(nr), np.arange(64), indexing="ij")
    dword = (wave + r * nw) * 64 + lane
    # LDS: the DMA of a round writes 64 dwords from its wave's base
    assert np.array_equal((wave * (64 // wpe) + r * nw * (64 // wpe)) * wpe + lane, dword)
    assert dword.max() < lps * wpe and lpw <= lps * wpe
    assert set(range(lpw)) <= set(dword.ravel().tolist())
    d = np.where(dword >= lpw, 0, dword)
    e, wd = d // wpe, d % wpe
    ey, ex = e // lx, e % lx
    assert ey.max() < ly
    for x0 in {0, (nx - 1) // tx * tx, (nx - 1) // tx // 2 * tx}:
        for y0 in {0, (ny - 1) // TY * TY, (ny - 1) // TY // 2 * TY}:
            gx, gy = (x0 + ex - R) % nx, (y0 + ey - R) % ny
            off = (gx + row * gy) * size + 4 * wd
            assert off.min() >= 0 and off.max() + 4 <= plane * size and off.max() < 2 ** 31
            # the cell that a thread at (tx, ty) reads at (dx, dy) from its centre is the grid's image of that neighbour
            cell = np.full(lps * wpe, -1, dtype=np.int64)
            cell[dword.ravel()] = off.ravel()
            ty_, tx_ = np.meshgrid(np.arange(TY), np.arange(tx), indexing="ij")
            for dx, dy in [(0, 0), (3, 0), (-3, 0), (0, 3), (0, -3), (3, 3), (-3, -3), (3, -3), (-3, 3), (1, 2)]:
                k = (ty_ + R + dy) * lx + (tx_ + R + dx)
                assert k.min() >= 0 and k.max() < lps
                want = ((x0 + tx_ + dx) % nx + row * ((y0 + ty_ + dy) % ny)) * size
                assert np.array_equal(cell[k * wpe], want)
                assert np.array_equal(cell[k * wpe + wpe - 1], want + 4 * (wpe - 1))
            # columns read without neighbours, the grid's first where the block is past it
            inside = (x0 + tx_ < nx) & (y0 + ty_ < ny)
            cx, cy = np.where(inside, x0 + tx_, 0), np.where(inside, y0 + ty_, 0)
            assert ((cx + row * cy) * size).max() + size <= plane * size
            assert (((cx + R) + (nx + 2 * R) * (cy + R)) * size).max() < 2 ** 31


@pytest.mark.parametrize("size", [4, 8])
@pytest.mark.parametrize("n", GRIDS)
def test_local_stage_writes_each_value_once(n, size):
    nx, ny, nz = n
    if nx * ny * nz > 4e6:
        ny = nz = 16
    line = 64 // size
    row = -(-nx // line) * line
    k, j, i = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    at = (i + row * j + row * ny * k).ravel()
    assert at.max() < row * ny * nz and np.unique(at).size == at.size
