"""Two contexts in one process: what one sets up does not change how the other's
launches run."""
import numpy as np
import pytest

from tests.systems import hairpin_design
from tis_amd.engine import MODE_EAGER, MODE_GRAPH, Engine

pytestmark = pytest.mark.gpu


def _engine(n, count):
    s, x = hairpin_design(50 + n, n)
    eng = Engine([s] * count, keys=list(range(count)), seed=5)
    for k in range(count):
        eng.set_coords(k, x)
    eng.langevin_init(tstep=0.05, rebuild_every=10)
    return eng


def test_windows_of_a_large_and_a_small_batch():
    """k_window's dynamic LDS is each batch's own: some 160 KB for the first
    context, 40 KB for the one created after it."""
    large, small, ref = _engine(107, 64), _engine(30, 2), _engine(107, 64)
    for steps in (15, 25):
        large.langevin_steps(steps, MODE_GRAPH)
        assert large.last_timing()["nlaunch"] == 1   # one k_window launch
        small.langevin_steps(steps, MODE_GRAPH)
        assert small.last_timing()["nlaunch"] == 1
        ref.langevin_steps(steps, MODE_EAGER)
        for k in (0, 1, 63):
            assert all(np.array_equal(large.get_state(k, w), ref.get_state(k, w)) for w in (0, 1, 2, 3))
    for e in (large, small, ref):
        e.close()
