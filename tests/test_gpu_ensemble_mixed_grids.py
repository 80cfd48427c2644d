"""Members whose grids differ (one to five cells per cutoff, a stencil larger
than the cell pass's segment table, crowded cells that workgroups share beside
sparse ones) advance in one ensemble, without lists, bit for bit as each does
alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def sort(W, n, cells, cutoff):
    sc = W.cell_sorting(n=n, L=16.0, cells=4, seed=n, cutoff=cutoff)
    return dict(sc, cells=[cells] * 3 if isinstance(cells, int) else cells)


def dpd(W, n, cells):
    sc = W.dpd_droplets(n=n, density=12.0, seed=n, radius=2.0, dt=1e-4)
    return dict(sc, cells=[cells] * 3, nspecies=0, fluxes=[], species=None)


def scenes(W, name):
    if name == "span3":
        return [sort(W, 800, 4, 3.5), sort(W, 1500, 16, 2.6), sort(W, 700, 4, 3.5)]
    if name == "parts":
        return [sort(W, 1000, 4, 3.5), sort(W, 1200, [32, 32, 8], 2.5), sort(W, 600, 4, 3.0)]
    if name == "shared":
        return [sort(W, 900, 4, 3.5), sort(W, 2000, 4, 3.5), sort(W, 1281, 4, 3.0), sort(W, 3000, 8, 3.0)]
    return [dpd(W, 1536, 5), dpd(W, 1700, 10), dpd(W, 1400, 4)]


@pytest.mark.parametrize("prec", [1, 0])
@pytest.mark.parametrize("name", ["span3", "parts", "shared", "dpd"])
def test_members_as_alone(gpu, tf, W, name, prec):
    alone = []
    for sc in scenes(W, name):
        eng, _ = W.build_engine(sc)
        eng.to_device(prec)
        eng.step(3)
        alone.append((eng.particles(), eng.energies()))
    engines = [W.build_engine(sc)[0] for sc in scenes(W, name)]
    ens = tf.Ensemble(engines, prec)
    ens.step(3)
    for k, (e, (p, en)) in enumerate(zip(engines, alone)):
        q = e.particles()
        for key in p:
            assert np.array_equal(q[key], p[key]), (k, key)
        assert e.energies() == en, k
    ens.close(download=False)
