"""Field solve by matrix products: grids with a side that the FFTs do not take (above 4080
and no power of two, or above 8192)."""
import math

import numpy as np
import pytest
from scipy import fft

import aieplace_amd as A
from aieplace_amd import api
from aieplace_amd.batch import BatchPlacer

PRECISIONS = [api.EP_PREC_FP32, api.EP_PREC_BF16X3, api.EP_PREC_FP16X3]
# relative size of what a product of two split operands drops
DROPPED = {api.EP_PREC_FP32: 0.0, api.EP_PREC_BF16X3: 2.0 ** -16, api.EP_PREC_FP16X3: 2.0 ** -21}


def fft_field(rho, wy_scale):
    """The oracle's field of a map, by scipy's FP64 FFTs (long grids)."""
    mx, my = rho.shape
    a = fft.dctn(rho, type=2) / (mx * my)  # 4 / (mx my) times the plain sums, scipy's being twice theirs per axis
    a[0] *= 0.5
    a[:, 0] *= 0.5
    wx, wy = np.pi * np.arange(mx)[:, None] / mx, np.pi * wy_scale * np.arange(my)[None, :] / my
    k2 = wx * wx + wy * wy
    k2[0, 0] = np.inf

    def cosines(x, axis):
        return 0.5 * (fft.dct(x, type=3, axis=axis) + np.take(x, [0], axis))

    def sines(x, axis):
        x = np.roll(x, -1, axis)  # the terms from 1 on; the constant one is 0
        return 0.5 * fft.dst(x, type=3, axis=axis)

    hx, hy = a * wx / k2, a * wy / k2
    return cosines(sines(hx, 0), 1), sines(cosines(hy, 0), 1)


def tolerance(mx, my, precision):
    """Three 2-D transforms whose sums round once per term, independently of each other
    (four standard deviations), and the dropped low parts of three products."""
    return 4 * 2.0 ** -24 * math.sqrt(1.5 * (mx + my)) + 3 * DROPPED[precision]


def placed(nl, p, seed):
    xl, yl, xh, yh = nl.die
    rng = np.random.default_rng(seed)
    pl = A.Placer(nl, p)
    pl.set_positions(xl + 0.7 * (xh - xl) * rng.random(pl.n_place), yl + 0.7 * (yh - yl) * rng.random(pl.n_place))
    return pl


@pytest.mark.parametrize("mx,my", [(16, 16), (48, 80), (7, 24)])
def test_reference_field_matches_oracle(oracle, mx, my):
    rho = np.random.default_rng(mx).random((mx, my))
    for got, want in zip(fft_field(rho, 0.7), oracle.field(rho, wy_scale=0.7)[1:]):
        assert np.abs(got - want).max() <= 1e-12 * np.abs(want).max()


# the long side in each direction, the other one as short as it goes, an FFT's or
# neither's; a power of two above the FFTs' largest
@pytest.mark.gpu
@pytest.mark.parametrize("mx,my", [(4112, 16), (16, 4112), (272, 4112), (4112, 4128), (16384, 16)])
def test_field_matches_reference(mx, my):
    print(f"case field products {mx} x {my}", flush=True)
    nl = A.generate("stdcell", seed=1, n_movable=2_000)
    p = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=mx, bins_y=my)
    with placed(nl, p, mx + my) as pl:
        fmap = pl.computeOverlaps()[0]
        fields = [pl.computeElectricFields(k) for k in PRECISIONS]
    bw, bh = (nl.die[2] - nl.die[0]) / mx, (nl.die[3] - nl.die[1]) / my
    want = fft_field(fmap.astype(np.float64) / (bw * bh), bw / bh)
    for k, got in zip(PRECISIONS, fields):
        err = [np.abs(g - e).max() / np.abs(e).max() for g, e in zip(got, want)]
        print(f"  precision {k}: {err[0]:.2e} {err[1]:.2e} (tolerance {tolerance(mx, my, k):.2e})", flush=True)
        assert max(err) <= tolerance(mx, my, k)
    assert not np.array_equal(fields[0][0], fields[1][0])  # the split forms are other arithmetic


@pytest.mark.gpu
@pytest.mark.parametrize("precision", PRECISIONS)
def test_evaluations_agree(oracle, precision):
    """The gradient of a product grid against the oracle, the field's reported error, and
    runs of either control, on one branch and on two, equal bit for bit."""
    from support import oracle_design
    mx, my = 4112, 16
    print(f"case evaluations products precision {precision}", flush=True)
    nl = A.generate("stdcell", seed=1, n_movable=3_000)
    p = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=mx, bins_y=my, precision=precision)
    d, _, _ = oracle_design(oracle, nl, p)
    with placed(nl, p, 3) as pl:
        x, y = pl.get_positions()
        g = pl.gradient(20.0, 3e-3)
        pl.overflow()
        assert max(pl.field_error(precision)) <= tolerance(mx, my, precision)
    o = d.gradient(x.astype(np.float64), y.astype(np.float64), p.target_density, 20.0, 3e-3)
    for k in ("gwx", "gwy", "fx", "fy", "gx", "gy"):
        assert np.abs(g[k] - o[k]).max() <= 2e-4 * np.abs(o[k]).max(), k
    out = []
    for graph, fork in ((0, 0), (1, 1), (1, 1 << 30)):
        p = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=mx, bins_y=my, precision=precision, use_graph=graph,
                            max_iters=9, fork_min_cells=fork)
        with A.Placer(nl, p) as pl:
            r = pl.run()
            out.append((r["iterations"], r["evals"], r["hpwl"], r["overflow"], *pl.get_positions()))
    assert out[0][0] == 9
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert np.array_equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", PRECISIONS)
@pytest.mark.parametrize("fork", [1, 1 << 30])
def test_batch_of_products_and_ffts(precision, fork):
    """A batch with grids on both paths reproduces its single-instance runs."""
    bins = [96, 4128, 256]
    print(f"case batch products and ffts precision {precision} fork {fork}", flush=True)
    nls = [A.generate("stdcell", seed=k + 1, n_movable=2_000) for k in range(len(bins))]
    p = A.placer_params(A.CONFIGS["stdcell_200k"], precision=precision, max_iters=4, fork_min_cells=fork)
    with BatchPlacer(nls, bins, p) as bp:
        bp.run()
        got = [bp.positions(i) for i in range(len(bins))]
    for nl, b, (x, y) in zip(nls, bins, got):
        q = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=b, bins_y=b, precision=precision, max_iters=4, use_graph=1)
        with A.Placer(nl, q) as pl:
            pl.run()
            sx, sy = pl.get_positions()
        assert np.array_equal(x, sx) and np.array_equal(y, sy), b


@pytest.mark.gpu
def test_side_above_65536():
    """A side whose matrix angles f (2 x + 1) pass 2^32.  Cells of one bin on every other
    bin around the middle: the map's spectrum sits at the highest frequencies.  The
    matrices take 83 GB of device memory."""
    mx, my = 68_000, 16
    print(f"case field products {mx} x {my}", flush=True)
    i, j = np.meshgrid(np.arange(32_000, 36_000, 2), np.arange(my), indexing="ij")
    on = np.random.default_rng(1).random(i.shape) < 0.5
    i, j = i[on], j[on]
    none = np.zeros(0, np.float32)
    nl = A.Netlist(die=(0, 0, mx, my), n_mov=len(i), w=np.ones(len(i)), h=np.ones(len(i)), x=i, y=j, net_start=np.zeros(1),
                   pin_cell=none, pin_dx=none, pin_dy=none)
    p = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=mx, bins_y=my, use_fillers=0)
    with A.Placer(nl, p) as pl:
        fmap = pl.computeOverlaps()[0]
        fields = [pl.computeElectricFields(k) for k in PRECISIONS]
    want = fft_field(fmap.astype(np.float64), 1.0)
    for k, got in zip(PRECISIONS, fields):
        err = [np.abs(g - e).max() / np.abs(e).max() for g, e in zip(got, want)]
        print(f"  precision {k}: {err[0]:.2e} {err[1]:.2e} (tolerance {tolerance(mx, my, k):.2e})", flush=True)
        assert max(err) <= tolerance(mx, my, k)
