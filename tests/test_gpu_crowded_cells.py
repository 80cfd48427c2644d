"""The cell pass of crowded systems (more than 20 particles per cell on
average), where a workgroup shares each cell, and its candidate staging:
force evaluations against the FP64 oracle.

Covered: mean occupancies just over the line, of several waves and of several
chunks of candidates, systems under the line with stencils of one, two and
three cells, non-periodic faces, radius transforms, DPD with a flux.
Positions lie on a grid of 2^-10 in cells whose size is a power of two, so
FP32 holds them exactly and both precisions evaluate the same state.
Tolerances: max |dF| / rms |F| <= 1e-10 (FP64) and 1e-5 (mixed, the suite's
bounds); number density 1e-12 and 1e-5 relative; pending flux 1e-10 and 1e-4
of its largest value.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def on_grid(sc, L, cells):
    x = np.floor(np.asarray(sc["x"]) / sc["dim"][0] * L * 1024.0) / 1024.0
    return dict(sc, dim=[float(L)] * 3, cells=[cells] * 3, x=np.clip(x, 0.0, L - 1.0 / 1024.0))


def scene(W, name):
    if name.startswith("mean"):
        n = dict(mean20=1300, mean31=2000, mean125=8000, mean312=20_000)[name]
        return on_grid(W.cell_sorting(n=n, L=16.0, cells=4, seed=n, cutoff=3.5), 16, 4)
    if name == "span2":
        return on_grid(W.cell_sorting(n=12_288, L=16.0, cells=8, seed=1, cutoff=3.5), 16, 8)
    if name == "span2_sparse":
        return on_grid(W.cell_sorting(n=3001, L=16.0, cells=8, seed=2, cutoff=3.5), 16, 8)
    if name == "span3_sparse":
        return on_grid(W.cell_sorting(n=5003, L=16.0, cells=16, seed=3, cutoff=2.5), 16, 16)
    if name == "one_particle_cells":
        return on_grid(W.cell_sorting(n=70, L=16.0, cells=4, seed=4, cutoff=3.5), 16, 4)
    if name == "walls":
        return on_grid(W.walled_morse(n=2500, L=16.0, cells=4, seed=5), 16, 4)
    if name == "radii":
        return on_grid(W.radius_mix(n=4096, density=1.0, seed=6), 16, 4)
    return on_grid(W.dpd_droplets(n=12_288, density=24.0, seed=7, radius=2.0), 8, 8)


@pytest.mark.parametrize("prec", [1, 0])
@pytest.mark.parametrize("name", ["mean20", "mean31", "mean125", "mean312", "span2", "span2_sparse", "span3_sparse",
                                  "one_particle_cells", "walls", "radii", "dpd_flux"])
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
    nd = np.abs(p["f"][:, 3] - o["f"][:, 3]) / o["f"][:, 3]
    assert nd.max() <= (1e-12 if prec else 1e-5)
    if sc["nspecies"]:
        q, r = p["species_q"], o["species_q"]
        assert np.abs(q - r).max() <= (1e-10 if prec else 1e-4) * np.abs(r).max()
    again = eng.particles()["f"]
    eng.set_launch(blocks=3)   # results do not depend on the launch shape
    eng.force()
    assert np.array_equal(eng.particles()["f"], again)
