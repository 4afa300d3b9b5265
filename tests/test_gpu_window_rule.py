"""Both sides of the rule that sends a batch of small systems to k_window or to
per-step launches: the same bits as eager mode, and the launches say which side
ran."""
import numpy as np
import pytest

from tests.systems import compact_allpairs, coulomb_chain, hairpin64, hairpin_design, two_chain_system
from tis_amd.engine import MODE_EAGER, MODE_GRAPH, Engine

pytestmark = pytest.mark.gpu


def _mix():
    # (398 beads leave few list rows in LDS: the crowded systems' entries past
    # them are read from memory)
    return ([hairpin64(0)] + [hairpin_design(50 + n, n) for n in (30, 43, 64, 65, 66, 107, 129, 133)]
            + [compact_allpairs(seed=20 + k) for k in range(2)]
            + [compact_allpairs(seed=9, ions=True), coulomb_chain(seed=4, n=100, box=50.0), two_chain_system()])


def _without_valence():
    return [hairpin_design(50 + n, n) for n in (30, 64, 107, 129)]


def _run(cases, mode, calls, rebuild):
    eng = Engine([s for s, _ in cases], seed=5)
    for k, (_, x) in enumerate(cases):
        eng.set_coords(k, x)
    eng.langevin_init(tstep=0.05, rebuild_every=rebuild)
    launches = 0
    for n in calls:
        eng.langevin_steps(n, mode)
        launches += eng.last_timing()["nlaunch"]
    out = [eng.get_state(k, w) for k in range(len(cases)) for w in (0, 1, 2, 3)]
    for k in range(0, len(cases), 7):
        out += [eng.pairs(k, 0), eng.pairs(k, 1)[0], eng.pairs(k, 2), *eng.term_status(k)]
    out.append(eng.energy_all())
    cnt = eng.counters()
    eng.close()
    return out, cnt, launches


@pytest.mark.parametrize("name,build,windows", [
    ("one long chain", lambda: [hairpin_design(179, 129)], False),
    ("one short chain", lambda: [hairpin_design(94, 44)], True),
    ("a few of every size", lambda: _without_valence() * 2, False),
    ("many of every size", lambda: _without_valence() * 64, True),
    ("every size and valence limits", lambda: _mix(), True),
    ("1,100 short chains", lambda: [hairpin_design(80, 30)] * 1100, False)])
@pytest.mark.parametrize("calls,rebuild", [((7, 13, 1, 30), 10), ((20, 3, 9), 7), ((55, 23), 0)])
def test_both_sides_equal_eager(name, build, windows, calls, rebuild):
    cases = build()
    print(f"[window rule] {name} calls {calls} rebuild {rebuild}", flush=True)
    a, ca, _ = _run(cases, MODE_EAGER, calls, rebuild)
    b, cb, launches = _run(cases, MODE_GRAPH, calls, rebuild)
    if rebuild > 0:   # (the trigger moves the line)
        assert (launches == len(calls)) == windows
    assert all(np.array_equal(u, v) for u, v in zip(a, b))
    assert ca == cb
