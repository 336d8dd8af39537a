"""CPU model of the resident kernels' tile links (k_tile_links in
csrc/engine_host.hip): the three tile ranges it finds for a tile must hold
every tile that owns a neighbour of one of the tile's cells, over full,
ragged and sparse anatomies, elongated along either end of the box order."""
import numpy as np
import pytest

NODES = [(-1, 0, 0), (0, -1, 0), (1, 0, 0), (0, 1, 0), (0, 0, -1), (0, 0, 1), (-1, -1, 0),
         (1, -1, 0), (1, 1, 0), (-1, 1, 0), (-1, 0, -1), (0, -1, -1), (1, 0, -1), (0, 1, -1),
         (-1, 0, 1), (0, -1, 1), (1, 0, 1), (0, 1, 1)]


def links(bi, plane, row):
    """Per tile three [first, last + 1) ranges, as the kernel computes them."""
    ntile = (bi.size + 63) // 64
    first = bi[::64]

    def upto(x):
        return int(np.searchsorted(first, x, side="right"))

    out = []
    for t in range(ntile):
        lo, hi = bi[64 * t], bi[min(64 * t + 63, bi.size - 1)]
        r = []
        for part in range(3):
            reach = row + 1 if part == 1 else row
            f = upto(lo + (part - 1) * plane - reach)
            e = upto(hi + (part - 1) * plane + reach)
            r.append((max(f - 1, 0), e) if e > 0 else (0, 0))
        out.append(r)
    return out


@pytest.mark.parametrize("dims,dens,seed", [((1, 1, 1), 1.0, 0), ((64, 1, 1), 1.0, 0),
                                            ((1, 1, 130), 1.0, 0), ((7, 8, 9), 1.0, 0),
                                            ((3, 5, 200), 1.0, 0), ((200, 5, 3), 0.8, 1),
                                            ((4, 90, 4), 0.6, 2), ((20, 21, 22), 0.15, 3),
                                            ((20, 21, 22), 0.9, 4), ((6, 6, 65), 0.02, 5)])
def test_every_neighbour_lies_in_a_linked_tile(dims, dens, seed):
    nx, ny, nz = dims
    rng = np.random.default_rng(seed)
    t = rng.random(dims) < dens
    if not t.any():
        t[0, 0, 0] = True
    x, y, z = np.nonzero(t)                       # box order: z fastest
    by, bz = ny + 2, nz + 2
    plane, row = by * bz, bz
    bi = ((x + 1) * plane + (y + 1) * row + (z + 1)).astype(np.int64)
    assert (np.diff(bi) > 0).all()
    tile_of = {int(b): k // 64 for k, b in enumerate(bi)}
    ln = links(bi, plane, row)
    reads = [set() for _ in ln]
    for k, b in enumerate(bi):
        for dx, dy, dz in NODES:
            n = tile_of.get(int(b + dx * plane + dy * row + dz))
            if n is not None:
                reads[k // 64].add(n)
    for k, r in enumerate(ln):
        covered = set()
        for a, e in r:
            assert 0 <= a <= e <= len(ln)
            covered.update(range(a, e))
        assert reads[k] <= covered
        # the wait is mutual: whom a tile reads also waits for it, so no tile
        # writes the box a neighbour still reads
        for n in reads[k]:
            assert any(a <= k < e for a, e in ln[n])
