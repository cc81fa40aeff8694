"""Kernels that share a launch against the same kernels on two branches."""
import numpy as np
import pytest

import aieplace_amd as A

pytestmark = pytest.mark.gpu


# sort blocks of 256 / 512 / 1024 cells, with the last block's cells missing or just
# begun; grids that are no multiple of the XCDs; fewer sort blocks than XCDs
@pytest.mark.parametrize("n", [8, 255, 2_049, 20_000, 81_921, 163_841, 327_681])
@pytest.mark.parametrize("fillers", [0, 1])
def test_shared_launches_equal_forked(n, fillers):
    """The same kernels in other launches: the trajectories are equal bit for bit."""
    print(f"case shared launches n={n} fillers={fillers}", flush=True)
    nl = A.generate("stdcell", seed=2, n_movable=n)
    out = []
    for fork in (1, 1 << 30):
        p = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=128, bins_y=128, use_fillers=fillers, use_graph=1,
                            max_iters=5, fork_min_cells=fork)
        with A.Placer(nl, p) as pl:
            r = pl.run()
            out.append((r["iterations"], r["evals"], r["hpwl"], r["overflow"], *pl.get_positions()))
    assert out[0][0] >= 1
    for a, b in zip(*out):
        assert np.array_equal(a, b)


def test_no_nets():
    """Without nets the net tiles and pin lists are empty: gradient and HPWL are of
    the density alone."""
    print("case no nets", flush=True)
    n = 300
    rng = np.random.default_rng(0)
    z = np.zeros(0, np.float32)
    nl = A.Netlist(die=(0, 0, 64, 64), n_mov=n, w=np.ones(n), h=np.ones(n), x=rng.random(n) * 64, y=rng.random(n) * 64,
                   net_start=np.zeros(1), pin_cell=z, pin_dx=z, pin_dy=z)
    p = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=32, bins_y=32, use_fillers=0)
    with A.Placer(nl, p) as pl:
        g = pl.gradient(1.0, 1.0)
    assert g["hpwl"] == 0.0
    assert not g["gwx"].any() and not g["gwy"].any()
    assert g["fx"].any() and g["fy"].any()
    # every movable cell has area 1 and no pins: the preconditioner is 1
    assert np.array_equal(g["gx"], -g["fx"]) and np.array_equal(g["gy"], -g["fy"])


# instances whose blocks end mid-grid: sort, net tile, density and cell grids that
# are no multiple of the XCDs
@pytest.mark.parametrize("counts", [(40,), (255, 1_025, 3_000), (9_000, 40, 20_001, 5_000, 700)])
def test_batch_shared_launches_equal_forked(counts):
    """As above for a batch's instances."""
    from aieplace_amd.batch import BatchPlacer
    print(f"case batch shared launches {counts}", flush=True)
    nls = [A.generate("stdcell", seed=3 + k, n_movable=n) for k, n in enumerate(counts)]
    out = []
    for fork in (1, 1 << 30):
        p = A.placer_params(A.CONFIGS["stdcell_200k"], max_iters=6, fork_min_cells=fork)
        bp = BatchPlacer(nls, [64] * len(counts), p)
        bp.run()
        out.append([a for i in range(len(counts)) for a in bp.positions(i)])
    for a, b in zip(*out):
        assert np.array_equal(a, b)


# limits on both sides of one and two batches of trials (8 in a single run, 4 in a
# batch), where the host stops queueing ahead
@pytest.mark.parametrize("limit", [1, 3, 4, 5, 7, 8, 9, 16, 17])
def test_iteration_limit(limit):
    """Device-controlled and batched runs stop at the limit where the host loop does, and
    a second run does nothing."""
    from aieplace_amd.batch import BatchPlacer
    print(f"case iteration limit {limit}", flush=True)
    nl = A.generate("stdcell", seed=4, n_movable=2_000)
    out = []
    for graph in (0, 1):
        p = A.placer_params(A.CONFIGS["stdcell_200k"], bins_x=64, bins_y=64, use_graph=graph, max_iters=limit)
        with A.Placer(nl, p) as pl:
            r = pl.run()
            assert r["iterations"] == limit
            assert pl.run()["evals"] == 0
            out.append((r["evals"], *pl.get_positions()))
    bp = BatchPlacer([nl], [64], p)
    bp.run()
    r = bp.results()
    assert r["iterations"][0] == limit
    out.append((r["evals"][0], *bp.positions(0)))
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert np.array_equal(a, b)
