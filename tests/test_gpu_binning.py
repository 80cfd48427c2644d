"""The binning: the scan of the cell counts on both sides of its forms (4,096
and 16,384 cells), the ordering of cells of 1 to 2,100 particles on both sides
of its groups (16) and of its key buffer (2,040), and the move of every
particle array, with species around its batches (4).

The forces of the binned state are compared with the FP64 oracle (they are
wrong if a particle is missing, twice there or in another cell), and the
records by particle id with the host's before the upload.  Positions lie on a
grid of 2^-10 in cells of a power of two, so FP32 holds them exactly.
Tolerances: max |dF| / rms |F| <= 1e-10 (FP64) and 1e-5 (mixed), the suite's
bounds; the records are equal.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def scene(W, n, cells, size, cutoff, seed, crowd=0):
    """n particles in cells of the given size, `crowd` more of them in one cell."""
    sc = W.cell_sorting(n=n + crowd, L=16.0, cells=4, seed=seed, cutoff=cutoff)
    dim = [float(c * size) for c in cells]
    x = np.asarray(sc["x"]) / sc["dim"][0] * dim
    x[n:] = size + x[n:] / np.array(dim) * size   # the cell (1, 1, 1)
    x = np.clip(np.floor(x * 1024.0) / 1024.0, 0.0, np.array(dim) - 1.0 / 1024.0)
    v = np.floor(np.random.default_rng(seed).normal(size=x.shape) * 1024.0) / 1024.0
    return dict(sc, dim=dim, cells=list(cells), x=x, v=v)


@pytest.mark.parametrize("prec", [1, 0])
@pytest.mark.parametrize("cells", [(16, 16, 16), (16, 16, 17), (16, 32, 32), (17, 31, 32)])
def test_cell_counts(gpu, tf, W, O, cells, prec):
    check(W, O, scene(W, 3001, cells, 1, 1.0, sum(cells)), prec)


@pytest.mark.parametrize("crowd", [1, 16, 17, 64, 2039, 2040, 2041, 2100])
def test_crowded_cell(gpu, tf, W, O, crowd):
    check(W, O, scene(W, 0, (4, 4, 4), 4, 3.5, crowd, crowd), 1)


def check(W, O, sc, prec):
    eng, pots = W.build_engine(sc)
    before = eng.particles()
    orc = O.Oracle(sc, pots)
    orc.force(8)
    eng.to_device(prec)
    eng.force()
    p, o = eng.particles(), orc.particles()
    for k in ("cid", "x", "v"):
        assert np.array_equal(p[k], before[k])
    f, g = p["f"][:, :3], o["f"][:, :3]
    scale = np.sqrt(np.mean(np.sum(g ** 2, axis=1)))
    assert np.linalg.norm(f - g, axis=1).max() <= (1e-10 if prec else 1e-5) * scale


@pytest.mark.parametrize("S", [1, 4, 5])
def test_species_move(gpu, tf, W, S):
    sc = scene(W, 3001, (8, 8, 8), 2, 2.0, S)
    sp = np.random.default_rng(S).integers(0, 1024, size=(3001, S)) / 1024.0
    sc = dict(sc, nspecies=S, species=sp)
    eng, _ = W.build_engine(sc)
    eng.to_device(0)
    eng.force()
    assert np.array_equal(eng.particles()["species"], sp)
