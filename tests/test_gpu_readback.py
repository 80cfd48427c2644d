"""Readback of the device state by particle id: the gather into host rows, for
sizes around its blocks (256 ids), chunks (2 MB) and the size several threads read (24 MB), in both precisions, after
reorderings, with species, and for members of an ensemble.

The reference is the host engine's own record before the upload: reading does
not change it, and on the FP32 path each coordinate is the host's rounded once
in the frame of the cell centre.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def host_record(eng, prec, tf):
    """Cell ids, positions and velocities of the engine on the host, as the device path stores them."""
    p = eng.particles()
    cdim, h, _ = eng.geometry()
    h = np.array(h)
    x, v = p["x"], p["v"]
    if prec == tf.PREC_MIXED:
        x = (x - 0.5 * h).astype(np.float32).astype(np.float64) + 0.5 * h
        v = v.astype(np.float32).astype(np.float64)
    loc = np.stack([p["cid"] // (cdim[1] * cdim[2]), p["cid"] // cdim[2] % cdim[1], p["cid"] % cdim[2]], axis=1)
    return p["cid"], x, v, loc * h + x


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("n,lists", [(1, False), (255, False), (256, True), (257, True), (20_001, False),
                                     (87_552, True), (300_007, True)])
def test_read_by_id(gpu, tf, W, n, lists, prec):
    L = max(9.0, float(n) ** (1.0 / 3.0))
    sc = W.cell_sorting(n=n, L=L, cells=int(L // 3.0), seed=n)
    sc["v"] = np.random.default_rng(n).normal(size=(n, 3))
    if lists:
        sc["verlet_skin"] = 0.4
    eng, _ = W.build_engine(sc)
    cid, x, v, xg = host_record(eng, prec, tf)
    eng.to_device(prec)
    eng.force()   # the slots are now in cell order
    for _ in range(2):
        p = eng.particles()
        assert np.array_equal(p["cid"], cid)
        assert np.array_equal(p["x"], x) and np.array_equal(p["v"], v)
        assert np.array_equal(eng.positions(), xg)
    # after steps: positions and records agree, and match what leaves the device
    eng.step(5)
    p, xg = eng.particles(), eng.positions()
    cdim, h, _ = eng.geometry()
    loc = np.stack([p["cid"] // (cdim[1] * cdim[2]), p["cid"] // cdim[2] % cdim[1], p["cid"] % cdim[2]], axis=1)
    assert np.array_equal(loc * np.array(h) + p["x"], xg)
    eng.from_device()
    q = eng.particles()
    for k in ("cid", "x", "v", "f"):
        assert np.array_equal(p[k], q[k])


def test_read_species(gpu, tf, W):
    sc = W.dpd_droplets(n=3000, seed=11)
    sc["species"] = np.random.default_rng(1).uniform(size=(3000, 1))
    eng, _ = W.build_engine(sc)
    eng.to_device(tf.PREC_FP64)
    eng.force()
    p = eng.particles()
    assert np.array_equal(p["species"], sc["species"])
    assert np.any(p["species_q"] != 0.0)
    eng.from_device()
    q = eng.particles()
    assert np.array_equal(p["species_q"], q["species_q"]) and np.array_equal(p["species"], q["species"])


def test_member_keeps_its_last_read(gpu, tf, W):
    """A member that leaves the ensemble without a download holds what was last read of it."""
    engines = [W.build_engine(W.cell_sorting(n=n, L=12.0, cells=4, seed=n))[0] for n in (500, 700, 900)]
    before = engines[2].particles()
    ens = tf.Ensemble(engines, tf.PREC_FP64)
    ens.step(3)
    first = engines[0].particles()
    engines[1].positions()
    e1 = engines[1].energies()
    second = engines[1].particles()
    ens.step(4)
    first = engines[0].particles()
    ens.step(2)
    ens.close(download=False)
    for got, want in ((engines[0].particles(), first), (engines[1].particles(), second), (engines[2].particles(), before)):
        for k in ("cid", "x", "v", "f"):
            assert np.array_equal(got[k], want[k])
    assert engines[1].energies() == e1
