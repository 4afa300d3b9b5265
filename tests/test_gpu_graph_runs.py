"""Captured graphs of per-step launches (batches with a system too large for
k_window): runs that stop for a list that overflows and resume, and the rebuild
counts, against eager and one-system-per-launch mode, bit for bit."""
import numpy as np
import pytest

from tests.systems import hairpin_design
from tis_amd.engine import MODE_EAGER, MODE_GRAPH, MODE_PLAIN, Engine

pytestmark = pytest.mark.gpu


def _run(mode, calls, rebuild, tight):
    # chains stretched by a third pull themselves together: the lists outgrow
    # a capacity that just fits the start
    cases = [(s, 1.3 * x) for s, x in (hairpin_design(50 + n, n) for n in (40, 64, 107, 170))]
    eng = Engine([s for s, _ in cases], seed=5)
    for k, (_, x) in enumerate(cases):
        eng.set_coords(k, x)
    eng.langevin_init(tstep=0.05, rebuild_every=rebuild)
    if tight:
        eng.list_capacity(max(int(np.bincount(eng.pairs(k, 0)[:, :2].ravel()).max()) for k in range(len(cases))))
    before = eng.counters()
    for n in calls:
        eng.langevin_steps(n, mode)
    if mode == MODE_GRAPH:
        assert eng.last_timing()["nlaunch"] > 1
    out = [eng.get_state(k, w) for k in range(len(cases)) for w in (0, 1, 2, 3)]
    out += [eng.pairs(k, w) for k in range(len(cases)) for w in (0, 2)]
    cnt = eng.counters()
    eng.close()
    return out, {k: cnt[k] - before[k] for k in cnt}


@pytest.mark.parametrize("calls,rebuild", [((120, 33), 10), ((61, 92), 7), ((153,), 0)])
def test_stopped_graphs_resume(calls, rebuild):
    print(f"[graph runs] calls {calls} rebuild {rebuild}", flush=True)
    ref, cref = _run(MODE_EAGER, calls, rebuild, False)
    assert cref["resumes"] == 0 and cref["steps"] == sum(calls)
    if rebuild:   # one before each multiple of the interval
        assert cref["rebuilds"] == -(-sum(calls) // rebuild)
    for mode in (MODE_GRAPH, MODE_EAGER, MODE_PLAIN):
        out, c = _run(mode, calls, rebuild, True)
        print("   ", mode, c, flush=True)
        assert c.pop("resumes") > 0
        # a resume repeats what the stopped launches had found: the systems that
        # the trigger had taken, the first system of one-system launches
        if rebuild == 0 or mode == MODE_PLAIN:
            c["rebuilds"] = cref["rebuilds"]
        assert c == {k: v for k, v in cref.items() if k != "resumes"}
        assert all(np.array_equal(u, v) for u, v in zip(out, ref))
