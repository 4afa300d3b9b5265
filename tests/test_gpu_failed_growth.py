"""Runs that stop because the neighbour lists may not grow any further: the call
fails, the state is the one after the last step that every system completed,
and what follows starts from there (no flag, count or buffer of the failed run
is left behind)."""
import numpy as np
import pytest

from tests.systems import hairpin_design
from tis_amd.engine import MODE_EAGER, MODE_GRAPH, MODE_PLAIN, Engine, TisError

pytestmark = pytest.mark.gpu


def _engine(sizes, rebuild):
    # chains stretched by a third pull themselves together: the lists outgrow
    # the capacity that fits the start, in different steps per system
    cases = [(s, 1.3 * x) for s, x in (hairpin_design(50 + n, n) for n in sizes)]
    eng = Engine([s for s, _ in cases], seed=5)
    for k, (_, x) in enumerate(cases):
        eng.set_coords(k, x)
    eng.langevin_init(tstep=0.05, rebuild_every=rebuild)
    return eng


def _fail(eng, n, steps, mode):
    """Lists limited to what they hold: a run of `steps` fails; the steps that
    every system completed."""
    most = 0
    for k in range(n):
        p = eng.pairs(k, 0)[:, :2].ravel()
        most = max(most, int(np.bincount(p).max()))
    eng.list_capacity(most)
    eng.list_limit(most)
    with pytest.raises(TisError, match="limit"):
        eng.langevin_steps(steps, mode)
    c = eng.counters()
    assert c["nb_overflow"] == 0 and c["run_completed"] == 0 and 0 <= c["steps"] < steps
    eng.list_limit(0)
    return c["steps"]


def _same(a, b, n, which=(0, 1, 2)):
    return all(np.array_equal(a.get_state(k, w), b.get_state(k, w)) for k in range(n) for w in which)


@pytest.mark.parametrize("rebuild", [10, 7, 0])
@pytest.mark.parametrize("mode", [MODE_EAGER, MODE_GRAPH, MODE_PLAIN])
def test_per_step_run_goes_on(mode, rebuild):
    sizes = (40, 64, 107, 170)   # 509 beads: no windows
    print(f"[failed growth] mode {mode} rebuild {rebuild}", flush=True)
    eng, ref = _engine(sizes, rebuild), _engine(sizes, rebuild)
    done = _fail(eng, len(sizes), 123, mode)
    print("    completed", done, flush=True)
    ref.langevin_steps(done, MODE_EAGER)
    assert _same(eng, ref, len(sizes))
    eng.langevin_steps(123 - done, mode)
    ref.langevin_steps(123 - done, MODE_EAGER)
    assert _same(eng, ref, len(sizes), (0, 1, 2, 3))
    assert all(np.array_equal(eng.pairs(k, 0), ref.pairs(k, 0)) for k in range(len(sizes)))
    assert eng.counters()["steps"] == 123
    eng.close(), ref.close()


@pytest.mark.parametrize("rebuild", [10, 7, 0])
def test_window_run_starts_again(rebuild):
    sizes = (40, 58, 50, 64)
    print(f"[failed growth] windows rebuild {rebuild}", flush=True)
    eng, ref = _engine(sizes, rebuild), _engine(sizes, rebuild)
    done = 0
    if rebuild == 10:   # in the second launch
        eng.langevin_steps(9, MODE_GRAPH)
        done = 9
    total = done + 123
    done = _fail(eng, len(sizes), total, MODE_GRAPH)
    print("    completed", done, flush=True)
    ref.langevin_steps(done, MODE_EAGER)
    assert _same(eng, ref, len(sizes))
    with pytest.raises(TisError, match="langevin_init"):
        eng.langevin_steps(5, MODE_GRAPH)
    for e in (eng, ref):
        e.neighbor(-1)
    assert all(np.array_equal(eng.force_sumup(k), ref.force_sumup(k)) for k in range(len(sizes)))
    for e, m in ((eng, MODE_GRAPH), (ref, MODE_EAGER)):
        e.langevin_init(tstep=0.05, rebuild_every=rebuild, step0=done, init_accel=False)
        e.langevin_steps(31, m)
    assert _same(eng, ref, len(sizes), (0, 1, 2, 3))
    eng.close(), ref.close()


def test_lists_that_cannot_be_built():
    """A list build that fails leaves no lists behind that later calls would
    take for whole ones."""
    eng, ref = _engine((64,), 1000), _engine((64,), 1000)
    most = int(np.bincount(eng.pairs(0, 0)[:, :2].ravel()).max())
    eng.list_capacity(most)
    eng.list_limit(most)
    for e in (eng, ref):
        e.langevin_steps(101, MODE_EAGER)   # (its only rebuild is that of the start)
    print(f"[failed growth] capacity {most}", flush=True)
    with pytest.raises(TisError, match="limit"):
        eng.neighbor(0)
    with pytest.raises(TisError, match="not built"):
        eng.pairs(0, 0)
    with pytest.raises(TisError, match="langevin_init"):
        eng.langevin_steps(1, MODE_EAGER)
    with pytest.raises(TisError, match="limit"):
        eng.force_sumup(0)
    eng.list_limit(0)
    ref.neighbor(0)
    assert np.array_equal(eng.force_sumup(0), ref.force_sumup(0))
    eng.close(), ref.close()
