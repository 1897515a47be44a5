"""The force pass with tabulated pairs in a batch of replicas with and without
tables, at row lengths around the pairs taken together: each equals its alone
run bit for bit, forked step included."""
import numpy as np
import pytest

from conftest import pos4_of

pytestmark = pytest.mark.gpu


def _desc(fmd, n, L, table, seed):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = (g * L / m + rng.uniform(0.0, 0.1, (n, 3))) % L
    r = np.linspace(0.6, 2.5, 300)
    rows = np.stack([r, r ** -9 - r ** -6, (9 * r ** -10 - 6 * r ** -7) / r], 1).astype(np.float32)
    lj = [1, 1, 0, 0, 0, 0, 1, 1] if table else [1, 1, 0.8, 1, 0.8, 1, 1, 1]
    return fmd.Desc(pos4_of(x, np.arange(n) % 2), L, np.asarray(lj, np.float32), ntypes=2, masses=[1.0, 1.5],
                    vel=rng.standard_normal((n, 3)), seed=seed,
                    tables=([-1, 0, 0, -1], [(0.6, 2.5, rows)]) if table else None)


@pytest.mark.parametrize("fork", ["0", "1"])
@pytest.mark.parametrize("n", [2, 5, 300, 1100])
def test_batch_with_and_without_tables(fmd, monkeypatch, n, fork):
    monkeypatch.setenv("FMD_STEP_FORK", fork)
    e = fmd.Engine(0)
    L = max(9.0, (n / 0.8) ** (1 / 3))
    descs = [_desc(fmd, n, L, t, 3 + k) for k, t in enumerate((True, False, True))]
    sids = [e.add(d) for d in descs]
    e.step(sids, 44)
    for d, s in zip(descs, sids):
        a = e.add(d)
        e.step(a, 44)
        for u, w in zip(e.state(a), e.state(s)):
            assert np.array_equal(u, w)
    e.close()
