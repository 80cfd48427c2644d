"""Near lists: between rebuilds the pair pass reads the list entries within
cutoff + a third of the skin, renewed when a particle has moved by half that.
They hold every pair within the cutoff, so trajectories are the cell pass's.

The sizes take both kernels that make them (one lane per particle from about
65,000, several below) and every number of lanes of the pair pass, with
remainders in the last block; 40 steps renew them several times.  FP64
trajectories agree to 1e-9 (sums of ~100 terms in another order, over 40
steps of contracting dynamics).  Forces at the same positions, with a
repulsive spring whose force at the cutoff is 20: a missing pair shows as a
jump of that size.  In FP32 the second engine's positions are rounded again
(1e-7), so a pair within that of the cutoff may differ (about 1 in 10^6
pairs, ~65 pairs a particle; 1 particle in 1000 allowed).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def engines(W, sc, skin):
    lists = W.build_engine(dict(sc, verlet_skin=skin))[0]
    cells = W.build_engine(sc)[0]
    return lists, cells


@pytest.mark.parametrize("n", [37, 1999, 20_003, 50_021, 140_001])
def test_fp64_trajectory(gpu, tf, W, n):
    L = max(9.0, float(n) ** (1.0 / 3.0))
    sc = W.cell_sorting(n=n, L=L, cells=max(3, int(L // 3.0)), seed=n)
    lists, cells = engines(W, sc, 0.4)
    for e in (lists, cells):
        e.to_device(tf.PREC_FP64)
        e.step(40)
    assert lists.verlet_state()[0] and not cells.verlet_state()[0]
    a, b = lists.positions(), cells.positions()
    d = a - b
    d -= L * np.round(d / L)
    assert np.abs(d).max() <= 1e-9
    e, f = lists.energies(), cells.energies()
    for k in e:
        assert abs(e[k] - f[k]) <= 1e-9 * max(1.0, abs(f[k]))


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n", [1999, 30_011, 140_001])
def test_no_pair_is_missing(gpu, tf, W, n, prec):
    L = float(n) ** (1.0 / 3.0)
    sc = W.cell_sorting(n=n, L=L, cells=int(L // 2.5), seed=n, cutoff=2.5)
    spring = dict(kind="harmonic", k=10.0, r0=4.5, min=0.0, max=2.5, tol=1e-3)
    sc["pots"] = [spring]
    sc["bind"] = [(0, 0, 0), (0, 1, 1), (0, 0, 1)]
    lists = W.build_engine(dict(sc, verlet_skin=0.5))[0]
    lists.to_device(prec)
    lists.step(20)
    for k in (1, 2, 3, 5, 4, 7):   # near lists of several ages
        lists.step(k)
        x = lists.positions()
        lists.step(1)              # its forces are those at x
        f = lists.particles()["f"]
        cells = W.build_engine(dict(sc, x=np.mod(x, L)))[0]
        cells.to_device(prec)
        cells.force()
        g = cells.particles()["f"]
        off = np.abs(f[:, :3] - g[:, :3]).max(axis=1)
        assert np.count_nonzero(off > 2.0) <= (max(2, n // 1000) if prec == 0 else 0)


def test_dpd_one_lane(gpu, tf, W):
    """DPD with one lane per particle: fast particles, so the near lists come and go."""
    sc = W.dpd_droplets(n=140_001, seed=3, dt=0.002)
    lists, cells = engines(W, sc, 0.4)
    for e in (lists, cells):
        e.to_device(tf.PREC_FP64)
        e.step(40)
    p, q = lists.particles(), cells.particles()
    L = sc["dim"][0]
    d = lists.positions() - cells.positions()
    d -= L * np.round(d / L)
    assert np.abs(d).max() <= 1e-9
    assert np.abs(p["v"] - q["v"]).max() <= 1e-8
    assert np.abs(p["species"] - q["species"]).max() <= 1e-9


@pytest.mark.parametrize("n", [1999, 140_001])
def test_no_room_behind_the_lists(gpu, tf, W, n):
    """A capacity that holds the lists but not the near lists behind them: the system keeps to the lists."""
    L = float(n) ** (1.0 / 3.0)
    sc = W.cell_sorting(n=n, L=L, cells=int(L // 3.0), seed=n)
    probe, cells = engines(W, sc, 0.4)
    probe.to_device(tf.PREC_FP64)
    probe.step(1)
    tight = probe.verlet_entries()[1] + 32
    lists = W.build_engine(dict(sc, verlet_skin=0.4, verlet_capacity=tight))[0]
    for e in (lists, cells):
        e.to_device(tf.PREC_FP64)
        for k in (1, 3, 36):
            e.step(k)
    assert lists.verlet_state()[2] < 1.5 * tight
    d = lists.positions() - cells.positions()
    d -= L * np.round(d / L)
    assert np.abs(d).max() <= 1e-9
