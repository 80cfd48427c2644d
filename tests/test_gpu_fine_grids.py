"""Grids of many cells per cutoff along x and y (the stencil has no limit there;
along z it is three cells): force evaluations against the FP64 oracle.

Covered: four to ten cells per cutoff, negative offsets over a periodic edge and
at walls, stencils larger than the cell pass's segment table (343 cells), whose
parts meet inside a chunk of candidates, for one wave per cell and for crowded
cells, with radii, DPD and a flux.  Positions lie on a grid of 2^-10 in cells
whose sizes are powers of two, so both precisions evaluate the same state.
Tolerances: max |dF| / rms |F| <= 1e-10 (FP64) and 1e-5 (mixed), the suite's
bounds; pending flux 1e-10 and 1e-4 of its largest value.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def on_grid(sc, h, cells):
    dim = np.array(cells, dtype=float) * h
    x = np.floor(np.asarray(sc["x"]) / sc["dim"] * dim * 1024.0) / 1024.0
    return dict(sc, dim=list(dim), cells=list(cells), x=np.clip(x, 0.0, dim - 1.0 / 1024.0))


def scene(W, name):
    def sort(n, h, cells, cutoff=2.5):
        return on_grid(W.cell_sorting(n=n, L=16.0, cells=4, seed=n, cutoff=cutoff), h, cells)
    if name == "x5":
        return sort(4001, [0.5, 2.0, 2.0], [32, 8, 8])
    if name == "y4":
        return sort(4003, [2.0, 0.5, 1.0], [8, 32, 16], cutoff=2.0)
    if name == "xy5":
        return sort(3001, [0.5, 0.5, 2.0], [32, 32, 8])
    if name == "x10_parts":
        return sort(6007, [0.25, 0.5, 1.0], [64, 32, 16])
    if name == "crowded_parts":
        return sort(21_701, [0.25, 1.0, 1.0], [21, 7, 7])
    if name == "walls_parts":
        sc = W.walled_morse(n=2500, L=16.0, cells=4, seed=5)
        return on_grid(dict(sc, cutoff=2.5), [0.25, 0.5, 1.0], [64, 32, 16])
    if name == "radii_parts":
        return on_grid(W.radius_mix(n=2048, density=0.5, seed=6), [0.25, 0.5, 1.0], [64, 32, 16])
    return on_grid(W.dpd_droplets(n=6000, density=12.0, seed=7, radius=2.0), [0.125, 0.25, 0.5], [64, 32, 16])


@pytest.mark.parametrize("prec", [1, 0])
@pytest.mark.parametrize("name", ["x5", "y4", "xy5", "x10_parts", "crowded_parts", "walls_parts", "radii_parts",
                                  "dpd_flux_parts"])
def test_forces(gpu, tf, W, O, name, prec):
    sc = scene(W, name)
    eng, pots = W.build_engine(sc)
    orc = O.Oracle(sc, pots)
    orc.force(8)
    eng.to_device(prec)
    eng.force()
    p, o = eng.particles(), orc.particles()
    assert np.array_equal(p["cid"], o["cid"])
    f, g = p["f"][:, :3], o["f"][:, :3]
    scale = np.sqrt(np.mean(np.sum(g ** 2, axis=1)))
    assert np.linalg.norm(f - g, axis=1).max() <= (1e-10 if prec else 1e-5) * scale
    if sc["nspecies"]:
        q, r = p["species_q"], o["species_q"]
        assert np.abs(q - r).max() <= (1e-10 if prec else 1e-4) * np.abs(r).max()


def test_noalloc(gpu, tf, W):
    sc = scene(W, "x10_parts")
    eng, _ = W.build_engine(sc)
    f, e = eng.force_noalloc(tf.PREC_FP64)
    eng.to_device(tf.PREC_FP64)
    eng.force()
    assert np.array_equal(eng.particles()["f"], f)


def test_z_is_limited(gpu, tf, W):
    eng, _ = W.build_engine(on_grid(W.cell_sorting(n=200, L=16.0, cells=4, seed=1, cutoff=2.5), [2.0, 2.0, 0.5], [8, 8, 32]))
    with pytest.raises(tf.TfgError) as e:
        eng.to_device(tf.PREC_FP64)
    assert e.value.code == tf.E_RANGE
