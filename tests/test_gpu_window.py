"""Batches of small systems run whole stretches of steps in one workgroup per
system (graph mode).  The per-step passes (eager mode) give the same bits:
state, forces, lists, hbond states, energies and counters, over fixed
intervals, calls that end between rebuilds, the displacement trigger, systems
at the limits of the layout, and a list capacity that has to grow inside the
run."""
import numpy as np
import pytest

from tis_amd.engine import MODE_EAGER, MODE_GRAPH, Engine
from tests.systems import compact_allpairs, coulomb_chain, hairpin64, hairpin_design, two_chain_system, valence_crowd

pytestmark = pytest.mark.gpu


def _run(cases, mode, calls, rebuild, cap=False):
    eng = Engine([s for s, _ in cases], seed=5)
    for k, (_, x) in enumerate(cases):
        eng.set_coords(k, x)
    eng.langevin_init(tstep=0.05, rebuild_every=rebuild)
    if cap:
        most = 0
        for k in range(len(cases)):
            p = eng.pairs(k, 0)[:, :2].ravel()
            most = max(most, int(np.bincount(p).max()) if len(p) else 0)
        eng.list_capacity(max(most, 1))
    for n in calls:
        eng.langevin_steps(n, mode)
    out = [eng.get_state(k, w) for k in range(len(cases)) for w in (0, 1, 2, 3)]
    for k in range(len(cases)):
        out += [eng.pairs(k, 0), eng.pairs(k, 1)[0], eng.pairs(k, 2), *eng.term_status(k)]
    out.append(eng.energy_all())
    cnt = eng.counters()
    eng.close()
    return out, cnt


def _mix():
    return ([hairpin64(0)] + [hairpin_design(50 + n, n) for n in (30, 43, 64, 65, 66, 107, 129, 149)]
            + [compact_allpairs(seed=20 + k) for k in range(2)] + [compact_allpairs(seed=9, ions=True),
                                                                   coulomb_chain(seed=4, n=100, box=50.0),
                                                                   two_chain_system()])


@pytest.mark.parametrize("calls,rebuild", [((40,), 10), ((7, 13, 1, 30, 5), 10), ((20, 3, 9), 7), ((130, 33), 0),
                                           ((520,), 100)])
def test_window_equals_per_step_passes(calls, rebuild):
    cases = _mix()
    print(f"[window] calls {calls} rebuild {rebuild} beads {[s.nmp for s, _ in cases]}", flush=True)
    a, ca = _run(cases, MODE_EAGER, calls, rebuild)
    b, cb = _run(cases, MODE_GRAPH, calls, rebuild)
    assert all(np.array_equal(u, v) for u, v in zip(a, b))
    assert ca == cb


def test_window_with_a_crowded_site():
    # 72 hbonds on each site of one G: sequences longer than a wave
    case = valence_crowd()
    print(f"[window crowd] beads {case[0].nmp}", flush=True)
    a, ca = _run([case], MODE_EAGER, (3,), 10)
    b, cb = _run([case], MODE_GRAPH, (3,), 10)
    assert ca["hb_deleted"] > 64 and ca == cb
    assert all(np.array_equal(u, v) for u, v in zip(a, b))


@pytest.mark.parametrize("rebuild", [10, 0])
def test_window_grows_the_lists(rebuild):
    # chains stretched by a third pull themselves together: the lists outgrow
    # a capacity that just fits the start, in different steps per system
    cases = [(s, 1.3 * x) for s, x in (hairpin_design(50 + n, n) for n in (40, 64, 107, 120))]
    print(f"[window capacity] rebuild {rebuild}", flush=True)
    a, ca = _run(cases, MODE_EAGER, (123, 30), rebuild, cap=True)
    b, cb = _run(cases, MODE_GRAPH, (123, 30), rebuild, cap=True)
    assert ca["resumes"] > 0 and cb["resumes"] > 0
    ca.pop("resumes"), cb.pop("resumes")   # each resume takes in what the stopped launch had found
    assert ca == cb
    assert all(np.array_equal(u, v) for u, v in zip(a, b))
