"""Calls in which almost every step rebuilds (thin skins): after a sample of 16
steps they send full steps only, 64 at a time, and must give the steps of calls
of one, bit for bit; so must the call in which such a system has settled."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("name", ["fast", "settling"])
def test_calls_equal_single_steps(gpu, tf, W, name, prec):
    if name == "fast":
        sc = dict(W.dpd_droplets(n=2000, seed=2, dt=0.005, noise="philox"), verlet_skin=0.02)
    else:
        sc = dict(W.cell_sorting(n=1500, L=11.5, cells=3, seed=6), verlet_skin=0.02)
    got, one = (W.build_engine(sc)[0] for _ in range(2))
    for eng in (got, one):
        eng.to_device(prec)
        assert eng.verlet_state()[0]
    for n in (20, 3, 150, 65):
        got.step(n)
        for _ in range(n):
            one.step(1)
        assert got.time == one.time
        assert got.verlet_state() == one.verlet_state()
        assert got.energies() == one.energies()
        a, b = got.particles(), one.particles()
        for k in a:
            assert np.array_equal(a[k], b[k]), k
    if name == "fast":   # the case that this is about
        assert one.verlet_state()[1] > 0.7 * one.time
