"""List overflows in a window launch whose systems do not all fit on the chip
at once: workgroups then start while another's overflow raises the stop flag,
and each has to take the flag as a whole.  The per-step passes (eager mode),
where no step is under way when it is raised, give the same bits."""
import numpy as np
import pytest

from tests.systems import hairpin_design
from tis_amd.engine import MODE_EAGER, MODE_GRAPH, Engine

pytestmark = pytest.mark.gpu


def _run(mode, rebuild):
    base = [hairpin_design(500 + n, n) for n in (40, 64, 50, 34, 61, 44, 58)]
    n = 600   # 256 CUs, one workgroup each
    # chains stretched by a third pull themselves together: the lists outgrow a
    # capacity that just fits the start, in different steps per system
    cases = [(base[k % 7][0], 1.3 * base[k % 7][1]) for k in range(n)]
    eng = Engine([s for s, _ in cases], keys=list(range(n)), seed=5)
    for k, (_, x) in enumerate(cases):
        eng.set_coords(k, x)
    eng.langevin_init(tstep=0.05, rebuild_every=rebuild)
    most = 0
    for k in range(n):
        p = eng.pairs(k, 0)[:, :2].ravel()
        most = max(most, int(np.bincount(p).max()) if len(p) else 0)
    eng.list_capacity(most)
    for steps in (90, 31):
        eng.langevin_steps(steps, mode)
    out = [eng.get_state(k, w) for k in range(n) for w in (0, 1, 2, 3)]
    for k in range(0, n, 37):
        out += [eng.pairs(k, 0), eng.pairs(k, 2)]
    out.append(eng.energy_all())
    cnt = eng.counters()
    eng.close()
    return out, cnt


@pytest.mark.parametrize("rebuild", [10, 0])
def test_overflow_while_workgroups_start(rebuild):
    print(f"[window stop] rebuild {rebuild}", flush=True)
    a, ca = _run(MODE_EAGER, rebuild)
    b, cb = _run(MODE_GRAPH, rebuild)
    print("   ", ca, cb, flush=True)
    assert ca["resumes"] > 0 and cb["resumes"] > 0
    assert all(np.array_equal(u, v) for u, v in zip(a, b))
    for c in (ca, cb):   # each resume takes in what the stopped launch had found
        c.pop("resumes"), c.pop("rebuilds")
    assert ca == cb
