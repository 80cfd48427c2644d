"""A pair at the very edge of the FP32 guard's band around a table end (b = 3
below the cutoff 3.5, distance 2.99998792): the pair loop and the rescan must
place it on the same side of the band, or it is dropped from both."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cells", [(20_000, 4), (12_288, 8)])
def test_no_pair_is_dropped(gpu, tf, W, O, n, cells):
    seed = n if cells == 4 else 1
    sc = W.cell_sorting(n=n, L=16.0, cells=cells, seed=seed, cutoff=3.5)
    sc["x"] = np.clip(np.floor(sc["x"] * 1024.0) / 1024.0, 0.0, 16.0 - 1.0 / 1024.0)   # exact in FP32
    nd = []
    for prec in (0, 1):
        eng, _ = W.build_engine(sc)
        eng.to_device(prec)
        eng.force()
        nd.append(eng.particles()["f"][:, 3])
    assert np.abs(nd[0] - nd[1]).max() <= 1e-5 * nd[1].min()   # one pair is 1e-3 of it
