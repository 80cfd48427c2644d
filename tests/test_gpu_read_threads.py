"""Reads of one ensemble from several host threads at once: every row equals
what one thread reads alone.  Members of different sizes make the shared pinned
buffers grow while another thread reads; the last sizes are read in chunks and
by several threads of the library itself (above 24 MB)."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def at_once(jobs):
    """Runs the jobs in a thread each, started together; returns their results."""
    gate = threading.Barrier(len(jobs))
    out = [None] * len(jobs)

    def run(k):
        gate.wait()
        try:
            out[k] = jobs[k]()
        except Exception as e:   # shown by the caller's comparison
            out[k] = e

    threads = [threading.Thread(target=run, args=(k,)) for k in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for o in out:
        if isinstance(o, Exception):
            raise o
    return out


def equal(a, b):
    return all(np.array_equal(a[k], b[k]) for k in b) if isinstance(b, dict) else np.array_equal(a, b)


def test_members(gpu, tf, W):
    sizes = [300, 30_011, 700, 90_001, 2000, 9001]
    engines = [W.build_engine(W.cell_sorting(n=n, L=max(9.0, n ** (1 / 3)), cells=3 if n < 1000 else int(n ** (1 / 3) // 3),
                                             seed=n))[0] for n in sizes]
    ens = tf.Ensemble(engines, tf.PREC_MIXED)
    ens.step(2)
    # the threads come first: the buffers are not there yet
    got = [at_once([e.positions if (k + r) % 2 else e.particles for k, e in enumerate(engines)]) for r in range(6)]
    want = [[e.positions() if (k + r) % 2 else e.particles() for k, e in enumerate(engines)] for r in range(2)]
    for r, row in enumerate(got):
        for k in range(len(sizes)):
            assert equal(row[k], want[r % 2][k]), (r, sizes[k])
    ens.close(download=False)
    for k, e in enumerate(engines):   # what was read of a member is what it holds
        assert equal(e.particles(), want[k % 2][k])
        assert equal(e.positions(), want[1 - k % 2][k])


@pytest.mark.parametrize("n", [2000, 300_007])
def test_one_engine_two_ways(gpu, tf, W, n):
    eng = W.build_engine(W.cell_sorting(n=n, L=n ** (1 / 3), cells=int(n ** (1 / 3) // 3), seed=n))[0]
    eng.to_device(tf.PREC_MIXED)
    eng.step(2)
    got = [at_once([eng.positions, eng.particles, eng.positions]) for _ in range(4)]
    x, p = eng.positions(), eng.particles()
    for a, b, c in got:
        assert equal(a, x) and equal(b, p) and equal(c, x)
