"""CPU model of the Jacobi block tiles (fs2d_jacobi.hpp): what a tile loads, how its
regions are placed, which neighbours the ring replaces, and what it writes.

Tiles of 32, 48 or 96 rows by 64 columns, m sweeps a launch.  A region's outer neighbours
are NaN here, so a cell that a launch writes from anything stale shows.  Each launch is
compared with m plain sweeps and ring updates of the whole grid; sums are taken in one
order, so the values are equal.  With margin 1 the tiles are placed for one sweep more, as
those that subtract the pressure's gradient afterwards: one cell around each written one
must be right too.  A batch's tiles are placed for its longest launch and may run fewer.
"""
from __future__ import annotations

import numpy as np
import pytest

COLS = 64
HEIGHTS = (32, 48, 96)


def tile_count(R, extent, m):
    return 1 if R <= extent else (R - 2 * m + extent - 2 * m - 1) // (extent - 2 * m)


def place(R, extent, m, t, tiles):
    """First cell of region t, and the first and last cell that it writes."""
    step = extent - 2 * m
    start = 0 if R <= extent else min(t * step, R - extent)
    return start, 1 if t == 0 else t * step + m, R - 2 if t == tiles - 1 else t * step + extent - 1 - m


def sweep(x, b, a, sign_tb, sign_lr):
    """One sweep of the whole grid and its ring."""
    y = x.copy()
    y[1:-1, 1:-1] = (b[1:-1, 1:-1] + a * (((x[:-2, 1:-1] + x[2:, 1:-1]) + x[1:-1, :-2]) + x[1:-1, 2:])) / (1 + 4 * a)
    y[0, 1:-1], y[-1, 1:-1] = sign_tb * y[1, 1:-1], sign_tb * y[-2, 1:-1]
    y[1:-1, 0], y[1:-1, -1] = sign_lr * y[1:-1, 1], sign_lr * y[1:-1, -2]
    return y


def run_tile(x, b, a, sign_tb, sign_lr, H, m, gi0, gj0):
    R = x.shape[0]
    rows = np.minimum(gi0 + np.arange(H), R - 1)
    cols = np.minimum(gj0 + np.arange(COLS), R - 1)
    X, B = x[np.ix_(rows, cols)].copy(), b[np.ix_(rows, cols)]
    left, right = gj0 == 0, gj0 + COLS >= R
    anywhere = R < H or (left and right)
    for s in range(m):
        p = np.pad(X, 1, constant_values=np.nan)
        north, south, west, east = p[:-2, 1:-1].copy(), p[2:, 1:-1].copy(), p[1:-1, :-2].copy(), p[1:-1, 2:].copy()
        if s > 0:
            if anywhere:  # ring cells by index
                gi, gj = gi0 + np.arange(H), gj0 + np.arange(COLS)
                north[gi == 1], south[gi == R - 2] = sign_tb * X[gi == 1], sign_tb * X[gi == R - 2]
                west[:, gj == 1], east[:, gj == R - 2] = sign_lr * X[:, gj == 1], sign_lr * X[:, gj == R - 2]
            else:  # known rows and lanes
                if gi0 == 0:
                    north[1] = sign_tb * X[1]
                if gi0 + H == R:
                    south[H - 2] = sign_tb * X[H - 2]
                if left:
                    west[:, 1] = sign_lr * X[:, 1]
                elif right:
                    east[:, COLS - 2] = sign_lr * X[:, COLS - 2]
        X = (B + a * (((north + south) + west) + east)) / (1 + 4 * a)
    return X


def launch(x, b, a, sign_tb, sign_lr, H, m, placed, margin):
    R = x.shape[0]
    out, written = np.full_like(x, np.nan), np.zeros(x.shape, int)
    ty, tx = tile_count(R, H, placed + margin), tile_count(R, COLS, placed + margin)
    around = np.full((R, R, 5), np.nan)  # each cell and its neighbours as its tile has them
    for i in range(ty):
        gi0, ilo, ihi = place(R, H, placed + margin, i, ty)
        for j in range(tx):
            gj0, jlo, jhi = place(R, COLS, placed + margin, j, tx)
            assert gi0 >= 0 and gj0 >= 0 and (R <= H or gi0 + H <= R) and (R <= COLS or gj0 + COLS <= R)
            X = run_tile(x, b, a, sign_tb, sign_lr, H, m, gi0, gj0)
            r, c = slice(ilo - gi0, ihi - gi0 + 1), slice(jlo - gj0, jhi - gj0 + 1)
            g = (slice(ilo, ihi + 1), slice(jlo, jhi + 1))
            out[g] = X[r, c]
            written[g] += 1
            if margin:
                p = np.pad(X, 1, constant_values=np.nan)
                for k, (di, dj) in enumerate(((0, 0), (-1, 0), (1, 0), (0, -1), (0, 1))):
                    around[g + (k,)] = p[ilo - gi0 + 1 + di : ihi - gi0 + 2 + di, jlo - gj0 + 1 + dj : jhi - gj0 + 2 + dj]
    assert np.all(written[1:-1, 1:-1] == 1) and written.sum() == (R - 2) ** 2
    return out, around


def check(R, H, m, placed, margin, sign_tb, sign_lr):
    rng = np.random.default_rng(R + 1000 * m + H)
    x, b, a = rng.standard_normal((R, R)), rng.standard_normal((R, R)), 0.3
    want = x
    for s in range(m):
        want = sweep(want, b, a, sign_tb, sign_lr)
    got, around = launch(x, b, a, sign_tb, sign_lr, H, m, placed, margin)
    assert np.array_equal(got[1:-1, 1:-1], want[1:-1, 1:-1]), (R, H, m)
    if margin:  # the ring is the cell itself there, whatever the tile holds
        for k, (di, dj) in enumerate(((0, 0), (-1, 0), (1, 0), (0, -1), (0, 1))):
            i = slice(2 if di < 0 else 1, -2 if di > 0 else -1)
            j = slice(2 if dj < 0 else 1, -2 if dj > 0 else -1)
            if R > 4:
                assert np.array_equal(around[i, j, k], np.roll(want, (-di, -dj), (0, 1))[i, j]), (R, H, m, k)


SIZES = sorted({3, 4, 5, 7, 20, 200, 333} | {e + d for e in (32, 48, 64, 96, 128, 160) for d in (-2, -1, 0, 1, 2, 17)})


@pytest.mark.parametrize("H", HEIGHTS)
@pytest.mark.parametrize("m", [1, 2, 3, 5, 8])
def test_tiles_are_plain_sweeps(H, m):
    for R in SIZES:
        check(R, H, m, m, 0, *((1, 1), (1, -1), (-1, 1))[R % 3])


@pytest.mark.parametrize("H", HEIGHTS)
@pytest.mark.parametrize("m", [1, 4, 8])
def test_tiles_with_a_margin_for_the_gradient(H, m):
    for R in SIZES:
        check(R, H, m, m, 1, 1, 1)


@pytest.mark.parametrize("H", HEIGHTS)
def test_tiles_placed_for_a_longer_launch(H):
    for R in SIZES:
        check(R, H, 6, 7, 0, 1, -1)


@pytest.mark.parametrize("extent", (*HEIGHTS, COLS))
def test_placement_at_every_size(extent):
    """Along one axis: cells 1 .. R - 2 are written once, each at least m from an end of its
    region that is not the grid's."""
    for m in range(1, 10):
        for R in range(3, 420):
            tiles, at = tile_count(R, extent, m), 1
            for t in range(tiles):
                start, lo, hi = place(R, extent, m, t, tiles)
                assert lo == at and hi >= lo
                assert start == 0 or lo - start >= m
                assert start + extent >= R or start + extent - 1 - hi >= m
                at = hi + 1
            assert at == R - 1, (R, m)
