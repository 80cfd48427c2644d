"""Steps of a call with neighbour lists: most run without the binning and the
build (light steps), which must not change anything.  A call of one step is a
full step, so n calls of one step are the reference, bit for bit: state,
energies, step counter and the number of rebuilds.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def scenes(W):
    sort = dict(W.cell_sorting(n=2000, L=12.6, cells=4, seed=1), verlet_skin=0.4)
    fast = dict(W.dpd_droplets(n=3000, seed=2, noise="philox"), verlet_skin=0.3)   # rebuilds every few steps
    fast["v"] = np.random.default_rng(3).normal(size=(3000, 3))
    bonded = dict(W.bonded_chains(nchains=60, beads=32, seed=4), verlet_skin=0.5, verlet_capacity=448)
    walls = dict(W.dpd_couette(n=3000, seed=5), verlet_skin=0.4)
    still = dict(W.cell_sorting(n=1500, L=11.5, cells=3, seed=6, dt=1e-7), verlet_skin=0.4)   # one build only
    return dict(sort=sort, fast=fast, bonded=bonded, walls=walls, still=still)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("name", ["sort", "fast", "bonded", "walls", "still"])
def test_light_steps_equal_full_steps(gpu, tf, W, name, prec):
    got, one = (W.build_engine(scenes(W)[name])[0] for _ in range(2))
    for eng in (got, one):
        eng.to_device(prec)
        assert eng.verlet_state()[0]
    for n in (2, 1, 37, 60):
        got.step(n)
        for _ in range(n):
            one.step(1)
        assert got.time == one.time
        assert got.verlet_state() == one.verlet_state()
        assert got.energies() == one.energies()
        a, b = got.particles(), one.particles()
        for k in a:
            assert np.array_equal(a[k], b[k]), k
    # a force pass between two calls leaves a rebuild to do
    for eng in (got, one):
        eng.force()
    assert got.energies() == one.energies()
    got.step(9)
    for _ in range(9):
        one.step(1)
    assert np.array_equal(got.positions(), one.positions())
    assert got.verlet_state() == one.verlet_state()


def test_light_steps_of_an_ensemble(gpu, tf, W):
    sizes = (700, 1900, 40)
    def make():
        return [W.build_engine(dict(W.cell_sorting(n=n, L=12.0, cells=4, seed=n), verlet_skin=0.4))[0] for n in sizes]
    a, b = make(), make()
    ea, eb = tf.Ensemble(a, tf.PREC_MIXED), tf.Ensemble(b, tf.PREC_MIXED)
    for n in (50, 23):
        ea.step(n)
        eb.step(n, use_graph=False)   # full steps
        for x, y in zip(a, b):
            assert np.array_equal(x.positions(), y.positions())
            assert x.verlet_state() == y.verlet_state() and x.energies() == y.energies()
    ea.close()
    eb.close()


def test_list_overflow_inside_a_call(gpu, tf, W):
    """A list over its capacity in a later step halts there, as with full steps: particles that all move to the centre."""
    def run(graph):
        sc = dict(W.cell_sorting(n=3000, L=20.0, cells=6, seed=7), verlet_skin=0.4, verlet_capacity=128)
        sc["types"] = [dict(t, dynamics=tf.NEWTONIAN) for t in sc["types"]]
        sc["v"] = 10.0 - sc["x"]
        eng = W.build_engine(sc)[0]
        ens = tf.Ensemble([eng], tf.PREC_FP64)
        ens.step(2, use_graph=graph)
        with pytest.raises(tf.TfgError) as e:
            ens.step(150, use_graph=graph)
        t = eng.time
        p = eng.particles()
        ens.close(download=False)
        return e.value.code, t, p
    ca, ta, pa = run(True)
    cb, tb, pb = run(False)
    assert ca == cb == tf.E_RANGE and ta == tb and ta > 4
    assert np.array_equal(pa["x"], pb["x"]) and np.array_equal(pa["cid"], pb["cid"])
