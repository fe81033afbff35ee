"""Tile binning at tile counts and capacities whose sort takes 8-bit and 9-bit
digits, an odd and an even number of passes, or one workgroup: keys, payloads
and ranges against a stable host sort of the emitted entries."""

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


# tiles_x * tiles_y gives the key bits above the 32 of the depth: 1 (33: 8-bit
# digits 5 passes, 9-bit 4), 5, 9 (41: 6 and 5), 13 (45: 6 and 5) and 14 (46:
# 6 each). Entries below and above 4096, the one-workgroup limit, and 2^17.
@pytest.mark.parametrize("tiles_x,tiles_y", [(1, 1), (5, 4), (20, 13), (120, 68), (128, 70)])
@pytest.mark.parametrize("n", [300, 3000, 60_000])
@pytest.mark.parametrize("digit", [8, 4])
def test_binner_digit_widths(gpu, tiles_x, tiles_y, n, digit):
    import splattar_amd as sa
    announce(f"binner {tiles_x}x{tiles_y} tiles, n {n}, digit {digit}")
    rng = np.random.default_rng(n + tiles_x)
    x0, y0 = rng.integers(0, tiles_x, n), rng.integers(0, tiles_y, n)
    x1, y1 = np.minimum(x0 + rng.integers(0, 3, n), tiles_x - 1), np.minimum(y0 + rng.integers(0, 2, n), tiles_y - 1)
    rects = np.stack([x0, y0, x1, y1], 1).astype(np.uint32)
    rects[rng.random(n) < 0.1] = (1, 1, 0, 0)  # no tile
    depth = rng.uniform(0.1, 9.0, n).astype(np.float32).view(np.uint32)
    depth[::7] = depth[0]  # ties
    keys, pays = [], []
    for i, (a, b, c, d) in enumerate(rects.astype(np.int64)):
        if c < a or d < b:
            continue
        ty, tx = np.meshgrid(np.arange(b, d + 1), np.arange(a, c + 1), indexing="ij")
        keys.append(((ty * tiles_x + tx).ravel().astype(np.uint64) << np.uint64(32)) | np.uint64(depth[i]))
        pays.append(np.full(ty.size, i, np.uint32))
    keys, pays = np.concatenate(keys), np.concatenate(pays)
    order = np.argsort(keys, kind="stable")
    keys, pays = keys[order], pays[order]
    e = keys.size
    b = sa.TileBinner(gpu, n, e + 5, tiles_x * tiles_y)
    b.rects.write(rects)
    b.depths.write(depth)
    b.encode(n, tiles_x, digit_bits=digit)
    assert int(b.entry_count().read()[0]) == e
    assert np.array_equal(b.sorted_keys().read(e), keys)
    assert np.array_equal(b.sorted_entries().read(e), pays)
    tile = (keys >> np.uint64(32)).astype(np.int64)
    want = np.zeros((tiles_x * tiles_y, 2), np.uint32)
    first = np.searchsorted(tile, np.arange(tiles_x * tiles_y), "left")
    last = np.searchsorted(tile, np.arange(tiles_x * tiles_y), "right")
    want[:, 0], want[:, 1] = np.where(last > first, first, 0), np.where(last > first, last, 0)
    assert np.array_equal(b.ranges.read(), want)
    assert not b.overflowed()
    b.close()
