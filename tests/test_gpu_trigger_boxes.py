"""Displacement-triggered rebuilds of every step: each is built from the positions
in front of its step and culled by the boxes of the same positions, so that its
pairs are the oracle's, however far the beads move in a step."""
import numpy as np
import pytest

import oracle
from tis_amd import topology as T
from tis_amd.engine import LIST_EXV, MODE_EAGER, Engine

pytestmark = pytest.mark.gpu


def _sorted(p):
    return p[np.lexsort(p.T[::-1])]


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_lists_of_chains_flying_apart(seed):
    """Two chains of two tiles each, 6 A further apart every step: boxes of the
    positions behind a step would miss the last pairs between them."""
    rng = np.random.default_rng(seed)
    s = T.build_rna_system([(T.random_sequence(rng, 43), []), (T.random_sequence(rng, 43), [])], neigh_margin=6.0,
                           name="apart")
    one = T.build_rna_system([(T.random_sequence(rng, 43), [])])
    a = T.compact_coords(one, rng, box=24.0, min_dist=2.6)
    a[:, 0] -= a[:, 0].max()
    x = np.concatenate([a, a * [-1.0, 1.0, 1.0] + [1.0, 0.0, 0.0]])
    v = np.zeros_like(x)
    v[:len(a), 0], v[len(a):, 0] = -64.0, 64.0
    eng = Engine([s], keys=[0], seed=11)
    eng.set_coords(0, x)
    eng.set_state(0, 1, v)
    eng.langevin_init(tstep=0.05, rebuild_every=0)
    eng.langevin_steps(1, MODE_EAGER)   # (no displacement yet in front of it)
    o = oracle.Oracle(s)
    between = []
    for step in range(3):
        x, before = eng.coords(0), eng.counters()["rebuilds"]
        eng.langevin_steps(1, MODE_EAGER)
        assert eng.counters()["rebuilds"] == before + 1
        o.neighbor(x)
        got, want = _sorted(eng.pairs(0, LIST_EXV)), _sorted(o.lists(0))
        between.append(int(((want[:, 0] < len(a)) & (want[:, 1] >= len(a))).sum()))
        print(f"[trigger boxes] seed {seed} step {step}: {len(want)} pairs, {between[-1]} between", flush=True)
        assert np.array_equal(got, want)
    assert between[0] > 0 and between[-1] == 0
    eng.close()
