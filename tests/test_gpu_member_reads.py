"""What was last read of a member is what its host engine holds when the
ensemble ends without a download, whatever changed the device state after the
read, and also without device memory to keep it in; such a read succeeds."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def members(W, sizes):
    return [W.build_engine(W.cell_sorting(n=n, L=max(9.0, n ** (1 / 3)), cells=max(3, int(n ** (1 / 3) // 3)), seed=n))[0]
            for n in sizes]


def equal(a, b):
    return all(np.array_equal(a[k], b[k]) for k in b)


@pytest.mark.parametrize("change", ["step", "force", "autotune", "nothing", "save"])
def test_kept_before_a_change(gpu, tf, W, tmp_path, change):
    engines = members(W, (600, 3000, 900))
    ens = tf.Ensemble(engines, tf.PREC_FP64)
    ens.step(2)
    first, energies = engines[1].particles(), engines[1].energies()
    engines[0].positions()
    if change == "step":
        ens.step(3)
    elif change == "force":
        ens.step(1)
        first, energies = engines[1].particles(), engines[1].energies()
        engines[2].force()
    elif change == "autotune":
        ens.autotune(1)
    elif change == "save":   # the host record becomes the later state
        ens.step(3)
        engines[1].save(str(tmp_path / "member.json"))
        first, energies = engines[1].particles(), engines[1].energies()
    ens.close(download=False)
    assert equal(engines[1].particles(), first)
    assert engines[1].energies() == energies
    if change == "nothing":
        host = members(W, (600, 3000, 900))
        assert equal(engines[2].particles(), host[2].particles())   # never read: as uploaded


def test_without_device_memory(gpu, tf, W):
    hip = tf.lib()   # the runtime's calls, through the library's own dependency
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def left():
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    engines = members(W, (500_000, 500_001))   # 88 MB to keep
    ens = tf.Ensemble(engines, tf.PREC_MIXED)
    ens.step(1)
    hold = []
    size = left()
    while size >= 4 << 20 and left() > 40 << 20:   # leave less than that
        size = min(size, left() - (32 << 20))
        p = ctypes.c_void_p()
        if hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)) == 0:
            hold.append(p)
        else:
            hip.hipGetLastError()
            size //= 2
    low = left()
    p = engines[1].particles()
    engines[0].positions()
    ens.step(1)
    for h in hold:
        assert hip.hipFree(h) == 0
    assert low < 80 << 20
    ens.step(1)
    ens.close(download=False)
    assert equal(engines[1].particles(), p)


def test_species_of_different_members(gpu, tf, W):
    """Members of 0, 1 and 3 species, one of them not read before the change."""
    def scene(n, S):
        sc = W.dpd_droplets(n=n, density=3.0, seed=n, radius=2.0)
        if S == 0:
            return dict(sc, nspecies=0, fluxes=[], species=None)
        return dict(sc, nspecies=S, species=np.random.default_rng(n).uniform(size=(n, S)))
    shapes = [(700, 1), (1500, 3), (600, 0), (900, 3)]
    engines = [W.build_engine(scene(n, S))[0] for n, S in shapes]
    host = W.build_engine(scene(*shapes[3]))[0].particles()
    ens = tf.Ensemble(engines, tf.PREC_FP64)
    ens.step(2)
    read = [e.particles() for e in engines[:3]]
    ens.step(2)
    ens.close(download=False)
    for e, want in zip(engines, read + [host]):
        assert equal(e.particles(), want)


def test_many_members(gpu, tf, W):
    """More members than one launch keeps (256), a part of them read."""
    engines = members(W, [200 + k % 7 for k in range(300)])
    ens = tf.Ensemble(engines, tf.PREC_MIXED)
    ens.step(1)
    read = {k: engines[k].particles() for k in (0, 31, 32, 130, 255, 256, 299)}
    ens.step(1)
    ens.close(download=False)
    for k, want in read.items():
        assert equal(engines[k].particles(), want), k
