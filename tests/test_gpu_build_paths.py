"""The list build's placement paths against the oracle's pair set: rows placed
by column from the hit masks, rows with more masks than that form holds, groups
that give the scan up (too many masks, or 32-bit rows that would meet them) and
the global scan, at group remainders and at boxes of 2 to 5 cells per axis;
one workgroup of four waves a tile (few groups) and one wave a tile (many)."""
import numpy as np
import pytest

from conftest import KG_LJ, pos4_of

pytestmark = pytest.mark.gpu

# (beads, box side): densities 0.3 to 4 at rc + skin = 2.8
SIZES = [(1, 9.0), (2, 9.0), (255, 8.6), (257, 8.6), (700, 8.5), (1500, 11.3), (2049, 14.2),  # 3 to 5 cells
         (2000, 8.5), (3000, 11.3), (2600, 9.0), (5000, 11.3), (900, 14.1), (1200, 5.7)]


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("n,L", SIZES)
def test_pairs_at_every_placement(fmd, engine, orc, monkeypatch, n, L, wide):
    if wide:
        monkeypatch.setenv("FMD_IDX32", "1")
    else:
        monkeypatch.delenv("FMD_IDX32", raising=False)
    rng = np.random.default_rng(n)
    L = np.float32(L)
    x = (rng.random((n, 3)) * L).astype(np.float32)
    x[:1] = 0.0
    if n > 8:  # on cell bounds, where the cell and the grid coordinate may disagree
        nx = int(L / np.float32(2.8))
        x[1:8] = (np.arange(7)[:, None] * (L / nx) % L).astype(np.float32)
        x[4] = np.nextafter(x[4], np.float32(0))
    bonds = None if n < 20 else [[8, k] for k in range(9, 16)]  # seven partners of one atom
    sid = engine.add(fmd.Desc(pos4_of(x), L, KG_LJ, force_cap=10.0, bonds=bonds,
                              bond_params=None if bonds is None else [[0.0, 1e3, 0.0, 1.0]]))
    p4, _, _ = engine.state(sid)
    excl = None if bonds is None else orc.exclusions(n, np.asarray(bonds, np.int32))
    ref = orc.pair_set(p4, L, np.float32(2.5) + np.float32(0.3), excl)
    assert np.array_equal(engine.pairs(sid), ref)
    engine.remove(sid)


def test_many_groups_build_the_rows_of_few(fmd, engine, orc):
    """A batch of more than 512 groups (one wave a tile) and the same system
    alone (four): the same rows, forces and trajectory bit for bit."""
    rng = np.random.default_rng(5)
    n, L = 12000, np.float32(24.2)
    g = np.stack(np.meshgrid(*[np.arange(23)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = (g * float(L) / 23 + 0.5 + rng.uniform(-0.08, 0.08, (n, 3))) % float(L)
    d = [fmd.Desc(pos4_of(x), L, KG_LJ, vel=rng.standard_normal((n, 3)), seed=k + 1) for k in range(12)]
    sids = [engine.add(k) for k in d]
    engine.step(sids, 45)
    alone = engine.add(d[0])
    engine.step(alone, 45)
    assert engine.rebuilds(alone) >= 3
    for a, b in zip(engine.state(sids[0]), engine.state(alone)):
        assert np.array_equal(a, b)
    assert np.array_equal(engine.pairs(sids[0]), engine.pairs(alone))
    engine.build_neighbors(alone)
    p4, _, _ = engine.state(alone)
    assert np.array_equal(engine.pairs(alone), orc.pair_set(p4, L, np.float32(2.5) + np.float32(0.3)))
    for s in sids + [alone]:
        engine.remove(s)


@pytest.mark.parametrize("n,L", [(3, 9.0), (257, 8.6), (1023, 10.6), (2049, 13.5), (16385, 27.0), (20480, 29.0), (20481, 29.0),
                                 (900, 60.0), (900, 91.0)])
def test_sort_in_one_workgroup(fmd, engine, orc, n, L):
    """The cell sort in the deciding workgroup (up to 20,480 atoms and 32,768
    cell keys) and by the five sort kernels (a batch with a replica above the
    limits): the same bits, and the exact pair set."""
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = (g * L / m + rng.uniform(0, 0.2, (n, 3))) % L
    x[0] = 0.0
    d = fmd.Desc(pos4_of(x), L, KG_LJ, vel=rng.standard_normal((n, 3)), seed=3, T=(1.0, 1.0))
    big = int(np.ceil(90000 ** (1 / 3)))
    gb = np.stack(np.meshgrid(*[np.arange(big)] * 3, indexing="ij"), -1).reshape(-1, 3) * 1.1
    other = fmd.Desc(pos4_of(gb), big * 1.1, KG_LJ, vel=rng.standard_normal((len(gb), 3)))
    a, b, c = engine.add(d), engine.add(d), engine.add(other)
    engine.step(a, 43)
    engine.step([b, c], 43)
    for u, w in zip(engine.state(a), engine.state(b)):
        assert np.array_equal(u, w)
    assert np.array_equal(engine.pairs(a), engine.pairs(b))
    assert engine.rebuilds(a) >= 3
    engine.step(a, 20 - 3)  # to the step of a forced rebuild at the latest
    engine.build_neighbors(a)
    p4, _, _ = engine.state(a)
    assert np.array_equal(engine.pairs(a), orc.pair_set(p4, np.float32(L), np.float32(2.5) + np.float32(0.3)))
    for s in (a, b, c):
        engine.remove(s)
