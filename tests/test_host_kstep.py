"""Host tables of the K-step 2D kernels with anchored regions (BZ_TILE_ANCHORED): the windows of stored cells
of a grid's regions partition it, and every monitor point is owned by the region that stores it."""
import numpy as np
import pytest

from beamz_amd import _native as N
from beamz_amd.simulation.engine import anchored_regions, kstep_owner_tables, xcd_order


def window(t, n, size, K):
    """First and last + 1 cell stored by region t along an axis of n cells, as the kernels compute them."""
    r0 = t * (size - 2 * K)
    return (r0 if t == 0 else r0 + K), min(n, r0 + size if r0 + size >= n else r0 + size - K)


@pytest.mark.parametrize("K,rh", [(8, 64), (12, 64), (16, 64), (15, 32), (31, 64)])
def test_anchored_windows_partition_every_axis_length(K, rh):
    for size in (64, rh):
        for n in list(range(2, 200)) + [600, 701, 1024]:
            g = anchored_regions(n, size, K)
            w = [window(t, n, size, K) for t in range(g)]
            assert w[0][0] == 0 and w[-1][1] == n, (n, w)
            assert all(a < b for a, b in w) and all(w[q][1] == w[q + 1][0] for q in range(g - 1)), (n, w)


@pytest.mark.parametrize("K,rh", [(8, 64), (12, 32), (31, 64)])
def test_anchored_points_have_the_owner_that_stores_them(K, rh):
    rng = np.random.default_rng(7)
    dims = np.array([(150, 90, 192), (37, 260, 64), (64, 64, 64), (301, 2, 320)], np.int64)   # (nx, ny, ld)
    rows = []
    for s, (nx, ny, _) in enumerate(dims):
        gx, gy = anchored_regions(nx, 64, K), anchored_regions(ny, rh, K)
        t = np.stack(np.meshgrid(np.arange(gx), np.arange(gy), indexing="xy"), -1).reshape(-1, 2)
        rows.append(np.concatenate([np.full((len(t), 1), s | N.TILE_ANCHORED), t], axis=1))
    tiles = xcd_order(np.concatenate(rows), per_wg=1)
    sim = rng.integers(0, len(dims), 600)
    jj, ii, comp = rng.integers(0, dims[sim, 1]), rng.integers(0, dims[sim, 0]), rng.integers(0, 3, 600)
    jj[:40], ii[:40] = 0, 0                                          # corners and far edges too
    jj[40:80], ii[40:80] = dims[sim[40:80], 1] - 1, dims[sim[40:80], 0] - 1
    pts = np.stack([sim, comp, jj * dims[sim, 2] + ii], axis=1)
    start, ents = kstep_owner_tables(tiles, pts, dims, K, rh)
    assert sorted(ents[:, 0].tolist()) == list(range(len(pts)))
    for q, (s, tx, ty) in enumerate(tiles):
        for p, code in ents[start[q]:start[q + 1]]:
            row, col, c = code >> 10, (code >> 2) & 255, code & 3
            assert (sim[p], comp[p]) == (s & ~N.TILE_ANCHORED, c)
            assert (ty * (rh - 2 * K) + row, tx * (64 - 2 * K) + col) == (jj[p], ii[p])
            nx, ny, _ = dims[sim[p]]
            x0, x1 = window(tx, nx, 64, K)
            y0, y1 = window(ty, ny, rh, K)
            assert x0 <= ii[p] < x1 and y0 <= jj[p] < y1
