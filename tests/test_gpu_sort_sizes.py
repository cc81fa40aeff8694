"""Tile sort and trial move at the sizes where their cells per thread change."""
import numpy as np
import pytest

import aieplace_amd as A
from aieplace_amd import api

pytestmark = pytest.mark.gpu


def maps_of(pl):
    out = [np.zeros(pl.bins, np.float32) for _ in range(2)]
    api.check(api.lib.ep_get_density(pl._ctx, api.fptr(out[0]), api.fptr(out[1]), None))
    return out


# 1 | 2 | 4 | 8 cells per thread begin at 256 x 160 times as many cells; one block,
# and the last of a block's cells missing
@pytest.mark.parametrize("n", [100, 255, 81_919, 81_921, 163_839, 163_840, 327_679, 327_681])
def test_counted_and_uncounted_sort_agree(n):
    """The maps of a trial (counted by the move) equal those of the same positions
    sorted afresh, and hold the movable cells' whole area."""
    print(f"case sort n={n}", flush=True)
    nl = A.generate("stdcell", seed=2, n_movable=n)
    p = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=128, bins_y=128, use_fillers=0, use_graph=1, max_iters=3)
    xl, yl, xh, yh = nl.die
    rng = np.random.default_rng(n)
    with A.Placer(nl, p) as pl:
        assert pl.n_place == n
        pl.set_positions(xl + rng.random(n) * (xh - xl), yl + rng.random(n) * (yh - yl))
        r = pl.run()
        assert r["iterations"] >= 1
        run_field, run_mov = maps_of(pl)
        field, mov, _, tau = pl.computeOverlaps()
    assert np.array_equal(run_field, field) and np.array_equal(run_mov, mov)
    area = float((nl.w[:n].astype(np.float64) * nl.h[:n]).sum())
    # 2^-24 relative per coordinate of up to 128 bins
    assert abs(mov.sum(dtype=np.float64) - area) <= 2.0 ** -15 * area
    assert tau == r["overflow"]


@pytest.mark.parametrize("n", [100, 5_000, 500_000, 800_000])
def test_totals_on_both_sides_of_the_one_block_reduction(n):
    """HPWL (a sum over every WA block's partial) against the net spans of the FP32
    pin positions in numpy."""
    print(f"case totals n={n}", flush=True)
    nl = A.generate("stdcell", seed=2, n_movable=n)
    p = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=512, bins_y=512)
    with A.Placer(nl, p) as pl:
        x, y = pl.get_positions()
        hpwl = pl.hpwl()
    span = 0.0
    for pos, fixed, off in ((x, nl.x, nl.pin_dx), (y, nl.y, nl.pin_dy)):
        at = np.where(nl.pin_cell < n, pos[np.minimum(nl.pin_cell, n - 1)], fixed[nl.pin_cell]) + off
        s = nl.net_start[:-1]
        span += (np.maximum.reduceat(at, s) - np.minimum.reduceat(at, s)).sum(dtype=np.float64)
    assert hpwl == pytest.approx(span, rel=1e-9)


# one super tile, several, a window cut to fit the LDS, none that fits
@pytest.mark.parametrize("mx,my,n", [(16, 16, 500), (48, 32, 2_000), (240, 400, 20_000), (640, 320, 90_000),
                                     (1024, 16, 30_000), (16, 2048, 3_000)])
def test_density_windows_match_oracle(oracle, mx, my, n):
    """Clustered and spread cells on grids with different density windows."""
    from support import oracle_design
    print(f"case density windows {mx} x {my}, {n} cells", flush=True)
    nl = A.generate("stdcell", seed=2, n_movable=n)
    p = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=mx, bins_y=my)
    d, x0, y0 = oracle_design(oracle, nl, p)
    xl, yl, xh, yh = nl.die
    rng = np.random.default_rng(n)
    spread = [(xl + rng.random(len(x0)) * (xh - xl)).astype(np.float32),
              (yl + rng.random(len(x0)) * (yh - yl)).astype(np.float32)]
    with A.Placer(nl, p) as pl:
        for x, y in ((x0, y0), spread):
            pl.set_positions(x, y)
            x, y = pl.get_positions()
            field, mov, _, _ = pl.computeOverlaps()
            omov = d.density(x.astype(np.float64), y.astype(np.float64), "exact", 0, d.n_mov)
            # every cell's edges round to 2^-24 of the grid side (in bins); a bin sums its cells' errors
            tol = 2.0 ** -22 * max(mx, my) * (xh - xl) / mx * (yh - yl) / my
            count = np.abs(omov).max() / ((xh - xl) / mx * (yh - yl) / my) + 4
            assert np.abs(mov - omov).max() <= tol * count * max(1.0, mx / my, my / mx)
            ofield = d.density(x.astype(np.float64), y.astype(np.float64), "stretched", 0, d.n_mov + d.n_fill)
            ofield += float(np.float32(p.target_density)) * d.density_fixed()
            assert abs(field.sum(dtype=np.float64) / ofield.sum() - 1) <= 1e-4
