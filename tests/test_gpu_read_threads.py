"""Reads of one engine's systems from several threads at once, the engine idle:
each gets its own system's arrays (of one range of the readback and of two)."""
import threading

import numpy as np
import pytest

from conftest import KG_LJ, pos4_of

pytestmark = pytest.mark.gpu


def test_reads_from_several_threads(fmd, engine):
    want = {}
    for n in (140000, 70001, 5000, 300):  # the largest first: the readback buffer has its size from then on
        rng = np.random.default_rng(n)
        m = int(np.ceil(n ** (1 / 3)))
        g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
        p4 = pos4_of(g * 1.1 + rng.uniform(0.0, 0.1, (n, 3)))
        v = rng.standard_normal((n, 3)).astype(np.float32)
        im = rng.integers(-3, 4, (n, 3)).astype(np.int32)
        want[engine.add(fmd.Desc(p4, max(m * 1.1 + 0.2, 9.0), KG_LJ, vel=v, image=im))] = (p4, v, im)
    wrong = []

    def read(sid):
        for _ in range(40):
            if not all(np.array_equal(u, w) for u, w in zip(engine.state(sid), want[sid])):
                wrong.append(sid)

    threads = [threading.Thread(target=read, args=(s,)) for s in list(want) * 2]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    for s in want:
        engine.remove(s)
