"""copyToBrick / copyFromBrick by 16-byte lanes: every element type, brick
counts off the wave's groups of bricks, arrays whose rows start off every
alignment, fields off 16 bytes, shuffled brick ids -- against numpy, byte for
byte, with everything outside the copied cells left alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NP = {0: np.uint64, 1: np.uint32, 2: np.uint16}


@pytest.mark.parametrize("dtype", [0, 1, 2], ids=["f64", "f32", "bf16"])
@pytest.mark.parametrize("nb,ghost,pad,offset,step", [
    ((1, 1, 1), 0, (0, 0, 0), 0, 512), ((3, 2, 1), 8, (1, 0, 2), 0, 512),
    ((4, 3, 2), 8, (8, 8, 8), 512, 1024), ((5, 1, 3), 0, (3, 1, 0), 1, 515),
    ((8, 2, 2), 8, (5, 0, 1), 3, 517), ((9, 3, 1), 8, (0, 7, 0), 8, 520),
    ((17, 1, 2), 0, (2, 2, 2), 0, 512), ((2, 9, 17), 8, (7, 3, 5), 2, 1030)])
def test_copies(gpu, dtype, nb, ghost, pad, offset, step):
    bk = gpu
    g = ghost // 8
    S = [n + 2 * g for n in nb]
    rng = np.random.default_rng(4)
    nbr = int(np.prod(S))
    grid = rng.permutation(nbr + 3)[:nbr].astype(np.uint32).reshape(S[2], S[1], S[0])
    info = bk.BrickInfo(np.zeros((nbr + 3, 27), np.uint32))
    ext = [8 * n + 2 * (p + ghost) for n, p in zip(nb, pad)]
    top = np.iinfo(NP[dtype]).max
    arr = rng.integers(0, top, (ext[2], ext[1], ext[0]), dtype=NP[dtype])
    fld = rng.integers(0, top, (nbr + 3, step), dtype=NP[dtype])
    inner = tuple(slice(p + ghost, p + ghost + 8 * n) for n, p in zip(nb[::-1], pad[::-1]))
    ids = grid[g:g + nb[2], g:g + nb[1], g:g + nb[0]].reshape(-1)
    # the field's storage a few elements longer, so an offset field fits
    buf = bk.DeviceBuffer(fld.nbytes + 64 * fld.itemsize + offset * fld.itemsize)
    buf.zero()
    d_arr, d_grid = bk.DeviceBuffer.from_array(arr), bk.DeviceBuffer.from_array(grid.reshape(-1))
    size = fld.itemsize
    buf.upload(fld.reshape(-1), offset=offset * size)
    st = bk.BrickStorage(buf, nbr + 3, step, dtype)
    br = bk.Brick(info, st, offset)
    dims = [8 * n for n in nb]
    bk.copyToBrick(dims, pad, (ghost,) * 3, d_arr, d_grid, br)
    want = fld.copy()
    cells = arr[inner].reshape(nb[2], 8, nb[1], 8, nb[0], 8).transpose(0, 2, 4, 1, 3, 5)
    want[ids, :512] = cells.reshape(-1, 512)
    got = buf.download(NP[dtype], fld.size, offset=offset * size).reshape(fld.shape)
    assert np.array_equal(got, want)
    # and back: from another field into the same array
    buf.upload(fld.reshape(-1), offset=offset * size)
    bk.copyFromBrick(dims, pad, (ghost,) * 3, d_arr, d_grid, br)
    back = arr.copy()
    back[inner] = fld[ids, :512].reshape(nb[2], nb[1], nb[0], 8, 8, 8).transpose(
        0, 3, 1, 4, 2, 5).reshape(dims[::-1])
    assert np.array_equal(d_arr.download(NP[dtype], arr.size).reshape(arr.shape), back)
