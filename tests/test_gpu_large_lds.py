"""The cell pass with the largest LDS layout: FP64, DPD and tables, a flux of
eight species and a stencil of three cells per cutoff take more than 64 KiB of a
compute unit's LDS per workgroup.  Forces and pending flux against the FP64
oracle (positions on a grid of 2^-10, tolerances of the suite)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [1, 0])
def test_forces(gpu, tf, W, O, prec):
    n, S = 2500, 8
    sc = W.dpd_droplets(n=n, density=3.0, seed=3, radius=2.0)
    L, h = 9.0, 0.375
    x = np.floor(np.asarray(sc["x"]) / sc["dim"][0] * L * 1024.0) / 1024.0
    morse = dict(kind="morse", d=1.0, a=4.0, r0=0.6, min=0.05, max=1.125, tol=1e-6, shifted=False)
    lj = dict(kind="lj", min=0.3, max=1.125, A=4e-4, B=4e-2, tol=1e-6)
    sc = dict(sc, dim=[L] * 3, cells=[int(L / h)] * 3, cutoff=1.125, x=np.clip(x, 0.0, L - 1.0 / 1024.0),
              pots=sc["pots"] + [morse, lj], bind=[(0, 0, 0), (0, 0, 1), (1, 1, 1), (0, 0, 2), (2, 1, 2), (0, 2, 2)],
              nspecies=S, species=np.random.default_rng(4).integers(0, 1024, size=(n, S)) / 1024.0,
              fluxes=[dict(kind=tf.FLUX_FICK, ta=a, tb=b, sa=k, sb=k, k=0.05 * (k + 1), decay=0.0, target=0.0, cutoff=0.0)
                      for k in range(S) for a in range(3) for b in range(a, 3) if (k + a + b) % 4 == 0])
    eng, pots = W.build_engine(sc)
    assert eng.geometry()[2] == [3, 3, 3]
    orc = O.Oracle(sc, pots)
    orc.force(8)
    eng.to_device(prec)
    eng.force()
    p, o = eng.particles(), orc.particles()
    f, g = p["f"][:, :3], o["f"][:, :3]
    scale = np.sqrt(np.mean(np.sum(g ** 2, axis=1)))
    assert np.linalg.norm(f - g, axis=1).max() <= (1e-10 if prec else 1e-5) * scale
    q, r = p["species_q"], o["species_q"]
    assert np.abs(q - r).max() <= (1e-10 if prec else 1e-4) * np.abs(r).max()
