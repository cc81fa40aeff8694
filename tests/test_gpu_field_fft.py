"""Field solve by FFTs (power-of-two grids) against the FP64 oracle."""
import math

import numpy as np
import pytest

import aieplace_amd as A
from aieplace_amd import api
from aieplace_amd.batch import BatchPlacer

pytestmark = pytest.mark.gpu


# every last-stage radix, one and many FFTs per block, the smallest and the
# largest side, both orientations of a long grid
@pytest.mark.parametrize("mx,my", [(16, 16), (32, 16), (16, 64), (128, 32), (64, 256), (512, 128), (1024, 16),
                                   (16, 2048), (4096, 16), (16, 8192), (8192, 32)])
def test_field_matches_oracle(oracle, mx, my):
    """Max-norm error within one rounding (2^-24) per butterfly level of the three
    2-D transforms; the same field in every precision."""
    print(f"case field fft {mx} x {my}", flush=True)
    nl = A.generate("stdcell", seed=1, n_movable=2_000)
    p = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=mx, bins_y=my)
    xl, yl, xh, yh = nl.die
    rng = np.random.default_rng(mx + my)
    with A.Placer(nl, p) as pl:
        pl.set_positions(xl + 0.7 * (xh - xl) * rng.random(pl.n_place), yl + 0.7 * (yh - yl) * rng.random(pl.n_place))
        fmap, _, _, _ = pl.computeOverlaps()
        fields = [pl.computeElectricFields(k) for k in (api.EP_PREC_FP32, api.EP_PREC_BF16X3, api.EP_PREC_FP16X3)]
    bw, bh = (xh - xl) / mx, (yh - yl) / my
    _, ex, ey = oracle.field(fmap.astype(np.float64) / (bw * bh), wy_scale=bw / bh)
    tol = 2.0 ** -24 * 3 * math.log2(mx * my)
    for got in fields:
        err = [np.abs(g - e).max() / np.abs(e).max() for g, e in zip(got, (ex, ey))]
        print(f"  {err[0]:.2e} {err[1]:.2e} (tolerance {tol:.2e})", flush=True)
        assert max(err) <= tol


def test_batch_mixes_ffts_and_products():
    """A batch with grids on both paths reproduces its single-instance runs."""
    bins = [32, 96, 256, 2048]
    nls = [A.generate("stdcell", seed=k + 1, n_movable=2_000) for k in range(len(bins))]
    p = A.placer_params(A.CONFIGS["stdcell_200k"], max_iters=6)
    with BatchPlacer(nls, bins, p) as bp:
        bp.run()
        got = [bp.positions(i) for i in range(len(bins))]
    for nl, b, (x, y) in zip(nls, bins, got):
        q = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=b, bins_y=b, max_iters=6, use_graph=1)
        with A.Placer(nl, q) as pl:
            pl.run()
            sx, sy = pl.get_positions()
        print(f"  bins {b}", flush=True)
        assert np.array_equal(x, sx) and np.array_equal(y, sy), b


def odd_terms(n):
    """Terms that the odd-radix stages of a length-n FFT add up one after another, at most."""
    odd = n // (n & -n)
    return sum(f for f in range(3, odd + 1, 2) for _ in range(12) if odd % f == 0 and (odd := odd // f)) / 2


# one odd prime, several in one stage and in two, long primes, one side a power of two,
# one long row or column, the largest side
@pytest.mark.parametrize("mx,my", [(48, 48), (80, 112), (240, 400), (336, 96), (1008, 16), (64, 272), (976, 128),
                                   (16, 2000), (48, 4048), (4080, 16), (272, 752)])
def test_mixed_field_matches_oracle(oracle, mx, my):
    """Sides that are no power of two: within one rounding per butterfly level and per
    term of an odd stage; the same field in every precision."""
    print(f"case field fft {mx} x {my}", flush=True)
    nl = A.generate("stdcell", seed=1, n_movable=2_000)
    p = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=mx, bins_y=my)
    xl, yl, xh, yh = nl.die
    rng = np.random.default_rng(mx + my)
    with A.Placer(nl, p) as pl:
        pl.set_positions(xl + 0.7 * (xh - xl) * rng.random(pl.n_place), yl + 0.7 * (yh - yl) * rng.random(pl.n_place))
        fmap, _, _, _ = pl.computeOverlaps()
        fields = [pl.computeElectricFields(k) for k in (api.EP_PREC_FP32, api.EP_PREC_BF16X3, api.EP_PREC_FP16X3)]
    bw, bh = (xh - xl) / mx, (yh - yl) / my
    _, ex, ey = oracle.field(fmap.astype(np.float64) / (bw * bh), wy_scale=bw / bh)
    tol = 2.0 ** -24 * 3 * (math.log2(mx * my) + odd_terms(mx) + odd_terms(my))
    for got in fields:
        err = [np.abs(g - e).max() / np.abs(e).max() for g, e in zip(got, (ex, ey))]
        print(f"  {err[0]:.2e} {err[1]:.2e} (tolerance {tol:.2e})", flush=True)
        assert max(err) <= tol


def test_batch_of_mixed_sides():
    """Batched solves of sides of every class equal the single instances' runs."""
    bins = [96, 64, 288, 352, 1056, 160]
    nls = [A.generate("stdcell", seed=k + 1, n_movable=1_500) for k in range(len(bins))]
    p = A.placer_params(A.CONFIGS["stdcell_200k"], max_iters=4)
    with BatchPlacer(nls, bins, p) as bp:
        bp.run()
        got = [bp.positions(i) for i in range(len(bins))]
    for nl, b, (x, y) in zip(nls, bins, got):
        q = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=b, bins_y=b, max_iters=4, use_graph=1)
        with A.Placer(nl, q) as pl:
            pl.run()
            sx, sy = pl.get_positions()
        print(f"  bins {b}", flush=True)
        assert np.array_equal(x, sx) and np.array_equal(y, sy), b


# powers of two with one and several rows per block, blocks past the last row, a long
# grid in each direction, sides that are none
@pytest.mark.parametrize("mx,my", [(16, 16), (48, 64), (16, 1024), (1024, 32), (256, 256), (400, 240), (64, 976),
                                   (16, 8192)])
def test_rows_make_the_maps(mx, my):
    """The map pass inside the field solve (gradient) against the one by itself
    (computeOverlaps): equal maps, an equal overflow up to the order of its FP64 sum,
    and cleared accumulators (a second pass gives the same)."""
    print(f"case rows maps {mx} x {my}", flush=True)
    nl = A.generate("stdcell", seed=1, n_movable=3_000)
    p = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=mx, bins_y=my)
    with A.Placer(nl, p) as pl:
        field, mov, _, tau = pl.computeOverlaps()
        for _ in range(2):
            g = pl.gradient(1.0, 1.0)
            made = [np.zeros(pl.bins, np.float32) for _ in range(2)]
            api.check(api.lib.ep_get_density(pl._ctx, api.fptr(made[0]), api.fptr(made[1]), None))
            assert np.array_equal(made[0], field) and np.array_equal(made[1], mov)
            assert g["tau"] == pytest.approx(tau, rel=mx * my * 2.0 ** -52)
        again = pl.computeOverlaps()
    assert np.array_equal(again[0], field) and np.array_equal(again[1], mov) and again[3] == tau


# long odd radices, two outputs per item: just enough items for a block's threads, not
# enough in a single FFT but in two, an odd and an even number of outputs
@pytest.mark.parametrize("mx,my", [(2032, 32), (1808, 48), (16, 3856), (4016, 16)])
def test_long_odd_radix_matches_oracle(oracle, mx, my):
    test_mixed_field_matches_oracle(oracle, mx, my)


# the longest row that makes the maps, and the ones past it on a short and a long grid
@pytest.mark.parametrize("mx,my", [(16, 4096), (16, 8192), (64, 8192)])
def test_maps_of_long_rows(mx, my):
    test_rows_make_the_maps(mx, my)
