"""Small systems in large boxes: the cell sort's scan with one to a thousand
passes of keys a workgroup (2^15 to 2^30 cell keys), alone and as one of a batch
of small replicas; the pair set against the oracle's, the same bits in the batch."""
import numpy as np
import pytest

from conftest import KG_LJ, pos4_of

pytestmark = pytest.mark.gpu


def _clumps(fmd, n, L, seed, **kw):
    """Clumps of 25 beads at a spacing of 1.1, some across the box's faces."""
    rng = np.random.default_rng(seed)
    g = np.stack(np.meshgrid(*[np.arange(3)] * 3, indexing="ij"), -1).reshape(-1, 3)[:25] * 1.1
    c = rng.uniform(0.0, L, ((n + 24) // 25, 3))
    c[0] = L - 1.0
    c[1] = 0.0
    # one clump a cell of 10, so that no two overlap
    c = np.unique(np.floor(c / 10.0), axis=0) * 10.0
    x = (c[:, None, :] + g[None] + rng.uniform(0.0, 0.05, (len(c), 25, 3))).reshape(-1, 3) % L
    return fmd.Desc(pos4_of(x), L, KG_LJ, vel=rng.standard_normal((len(x), 3)), seed=seed, **kw)


@pytest.mark.parametrize("n,L", [(300, 80.0), (3000, 91.0), (3000, 190.0), (3000, 357.0), (200, 700.0), (3000, 1440.0)])
def test_pairs_in_a_large_box(fmd, engine, orc, n, L):
    sid = engine.add(_clumps(fmd, n, L, 3))
    for _ in range(2):
        p4, _, _ = engine.state(sid)
        ref = orc.pair_set(p4, np.float32(L), np.float32(2.5) + np.float32(0.3))
        assert len(ref) > 100 and np.array_equal(engine.pairs(sid), ref)
        engine.step(sid, 41)
        engine.build_neighbors(sid)
    assert engine.rebuilds(sid) >= 5
    engine.remove(sid)


@pytest.mark.parametrize("nr,L", [(1, 190.0), (40, 190.0), (40, 370.0), (300, 190.0)])
def test_large_box_in_a_batch(fmd, nr, L):
    e = fmd.Engine(0)
    d = [_clumps(fmd, 400, 40.0 + k % 7, k) for k in range(nr)] + [_clumps(fmd, 2000, L, 77)]
    sids = [e.add(k) for k in d]
    e.step(sids, 45)
    for k in (0, nr - 1, nr):
        alone = e.add(d[k])
        e.step(alone, 45)
        assert e.rebuilds(alone) >= 3
        for u, w in zip(e.state(alone), e.state(sids[k])):
            assert np.array_equal(u, w)
        assert np.array_equal(e.pairs(alone), e.pairs(sids[k]))
    e.close()
