"""The end of a step writes the flags of the next one (whether it is observed,
whether its start is prepared): a run in which they change at every step equals,
bit for bit, the same steps taken one call at a time (where every step is
observed and prepared anew).  Replicas of one chunk of partials, of several
summed in the boundary's workgroup, and of more."""
import numpy as np
import pytest

from conftest import KG_LJ, pos4_of

pytestmark = pytest.mark.gpu

STEPS = 24


def _desc(fmd, n, ens, freq, stress):
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1 / 3)))
    L = max(1.1 * m, 9.0)
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    x = (g * L / m + rng.uniform(0.0, 0.1, (n, 3))) % L
    kw = dict(ensemble=ens, T=(1.0, 1.2), P=(0.0, 1.0), Tdamp=0.5, Pdamp=1.0) if ens else dict(T=(1.0, 1.2))
    return fmd.Desc(pos4_of(x), L, KG_LJ, vel=rng.standard_normal((n, 3)), seed=n, thermo_freq=freq,
                    stress_freq=stress, nsteps=STEPS, **kw)


@pytest.mark.parametrize("ens", [0, 1, 2])
@pytest.mark.parametrize("n", [70, 16385, 70000])
def test_flags_that_change_every_step(fmd, engine, n, ens):
    d = _desc(fmd, n, ens, 2, 4)
    a, b = engine.add(d), engine.add(d)
    engine.step(a, STEPS)
    for _ in range(STEPS):
        engine.step(b, 1)
    for u, w in zip(engine.state(a), engine.state(b)):
        assert np.array_equal(u, w)
    rows, lost = engine.drain_thermo(a)
    assert lost == 0 and [r["step"] for r in rows] == list(range(2, STEPS + 1, 2))
    assert (rows, lost) == engine.drain_thermo(b)
    assert engine.box(a) == engine.box(b)
    ta, tb = engine.thermostat(a), engine.thermostat(b)
    assert all(np.array_equal(ta[k], tb[k]) for k in ta), (ta, tb)
    for s in (a, b):
        engine.remove(s)


@pytest.mark.parametrize("freq", [1, 3])
def test_batch_with_observed_and_unobserved_steps(fmd, engine, freq):
    """Replicas whose observed steps fall differently, in one batch and alone."""
    descs = [_desc(fmd, 300 + k, k % 3, freq * (1 + k % 2), 0 if k % 2 else 3) for k in range(9)]
    sids = [engine.add(d) for d in descs]
    engine.step(sids, STEPS)
    for d, s in zip(descs, sids):
        a = engine.add(d)
        engine.step(a, STEPS)
        for u, w in zip(engine.state(a), engine.state(s)):
            assert np.array_equal(u, w)
        assert engine.drain_thermo(a) == engine.drain_thermo(s)
        engine.remove(a)
    for s in sids:
        engine.remove(s)


@pytest.mark.parametrize("n", [16385, 40000, 65000])
def test_sums_of_every_step_and_of_the_last(fmd, engine, n):
    """Langevin replicas of two to four chunks: observed at every step (the chunks
    summed by a launch of their own) and at the last only (in the boundary's
    workgroup), the same state and the same last record, resumed ones included."""
    descs = [_desc(fmd, n, 0, 1, 0), _desc(fmd, n, 0, STEPS, 0)]
    sids = [engine.add(d) for d in descs]
    for s in sids:
        engine.step(s, STEPS - 4)
    sids.append(engine.resume(engine.snapshot(sids[0])))
    for s in sids:
        engine.step(s, 4)
    last = [engine.drain_thermo(s)[0][-1] for s in sids]
    assert last[0] == last[1] == last[2] and last[0]["step"] == STEPS
    for s in sids[1:]:
        for u, w in zip(engine.state(sids[0]), engine.state(s)):
            assert np.array_equal(u, w)
    for s in sids:
        engine.remove(s)
