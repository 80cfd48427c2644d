"""Force evaluations on both sides of the density from which workgroups share
crowded cells: 14 particles per cell up to 1,024 cells, 16 up to 2,048, 18 up
to 4,096, 20 above.  Compared with the FP64 oracle; positions lie on a grid of 2^-10 in
cells of a power of two, so FP32 holds them exactly.  Tolerances: max |dF| /
rms |F| <= 1e-10 (FP64) and 1e-5 (mixed), the suite's bounds.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def on_grid(sc, h, cells):
    dim = np.array(cells, dtype=float) * h
    x = np.floor(np.asarray(sc["x"]) / sc["dim"] * dim * 1024.0) / 1024.0
    return dict(sc, dim=list(dim), cells=list(cells), x=np.clip(x, 0.0, dim - 1.0 / 1024.0))


@pytest.mark.parametrize("prec", [1, 0])
@pytest.mark.parametrize("kind", ["morse", "radii", "dpd_flux"])
@pytest.mark.parametrize("cells,mean", [((4, 4, 4), 14), ((8, 8, 16), 14), ((8, 8, 17), 16), ((8, 16, 16), 16),
                                        ((8, 16, 17), 18), ((16, 16, 16), 18), ((16, 16, 17), 20)])
def test_both_sides(gpu, tf, W, O, cells, mean, kind, prec):
    ncells = int(np.prod(cells))
    for n in (mean * ncells, mean * ncells + 1):
        if kind == "morse":
            sc = on_grid(W.cell_sorting(n=n, L=16.0, cells=4, seed=n, cutoff=1.0), 1.0, cells)
        elif kind == "radii":
            sc = on_grid(W.radius_mix(n=n, density=0.5, seed=n), 4.0, cells)
        else:
            sc = on_grid(W.dpd_droplets(n=n, density=float(mean), seed=n, radius=2.0), 1.0, cells)
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
