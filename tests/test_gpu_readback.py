"""Readback by global id in ranges of 131,072 atoms, blocks of 256: the state of
a new system is its input (whatever order the cell sort put the atoms in), any
of the arrays alone, and the forces of a system of more than one range agree
with the FP64 oracle."""
import ctypes as C

import numpy as np
import pytest

from conftest import KG_LJ, pos4_of, rel_err_floor

pytestmark = pytest.mark.gpu


def _lattice(n, seed=1):
    rng = np.random.default_rng(seed)
    m = int(np.ceil(n ** (1 / 3)))
    a = 1.1
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = (g * a + rng.uniform(0.0, 0.1, (n, 3)))[rng.permutation(n)].astype(np.float32)
    return pos4_of(x), np.float32(max(m * a + 0.2, 9.0)), rng


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 5000, 131071, 131072, 131073, 262144, 262401])
def test_state_is_the_input(fmd, engine, n):
    p4, L, rng = _lattice(n)
    v = rng.standard_normal((n, 3)).astype(np.float32)
    im = rng.integers(-3, 4, (n, 3)).astype(np.int32)
    sid = engine.add(fmd.Desc(p4, L, KG_LJ, vel=v, image=im))
    for got, want in zip(engine.state(sid), (p4, v, im)):
        assert np.array_equal(got, want)
    for k in range(3):  # one array alone
        out = [np.full_like(a, 7) for a in (p4, v, im)]
        ptr = [a.ctypes.data_as(C.POINTER(C.c_int32 if q == 2 else C.c_float)) if q == k else None
               for q, a in enumerate(out)]
        assert fmd.lib().fmd_get_state(engine.h, sid, *ptr) == 0
        assert np.array_equal(out[k], (p4, v, im)[k])
        assert all(np.all(out[q] == 7) for q in range(3) if q != k)
    engine.remove(sid)


@pytest.mark.parametrize("n", [257, 131073])
def test_forces_by_global_id(fmd, engine, orc, n):
    p4, L, _ = _lattice(n)
    sid = engine.add(fmd.Desc(p4, L, KG_LJ))
    f, vir, pe = engine.forces(sid)
    f8, v8 = orc.forces_f64(p4, L, KG_LJ, terms=1)
    floor = np.sqrt(np.mean(np.sum(f8[:, :3] ** 2, axis=1)))
    assert rel_err_floor(f[:, :3], f8[:, :3], floor) < 1e-5
    assert abs(pe - f8[:, 3].sum()) <= 1e-5 * abs(f8[:, 3].sum())
    engine.remove(sid)


def test_thermo_rows_across_the_ring_end(fmd, engine):
    """Records drained in one run of the ring and in two."""
    p4, L, rng = _lattice(300)
    d = fmd.Desc(p4, L, KG_LJ, vel=rng.standard_normal((300, 3)), thermo_freq=1)
    sid, other = engine.add(d), engine.add(d)
    engine.step(sid, 4000)
    head, lost = engine.drain_thermo(sid)
    assert lost == 0 and [r["step"] for r in head] == list(range(1, 4001))
    engine.step(sid, 200)  # past the ring's 4,096 records
    tail, lost = engine.drain_thermo(sid)
    assert lost == 0 and [r["step"] for r in tail] == list(range(4001, 4201))
    engine.step(other, 4000)
    engine.drain_thermo(other)
    for k in range(4):
        engine.step(other, 50)
        rows, _ = engine.drain_thermo(other)
        assert rows == tail[50 * k:50 * k + 50]
    for s in (sid, other):
        engine.remove(s)
