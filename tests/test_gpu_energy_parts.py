"""energy_sumup shared out over blocks (one per 256 beads or two chunk
pairs of 64 charges): systems at the edges of that split against the FP64
oracle, and the same bits alone, in the batch call and in a set call."""
import numpy as np
import pytest

import oracle
from tis_amd.engine import Engine
from tests.systems import compact_allpairs, coulomb_chain, hairpin_design, small_ions_box

pytestmark = pytest.mark.gpu


def _cases():
    # nt - 1 charges and 3 nt - 1 beads: one and two chunks, 254 / 257 beads,
    # 1 -> 3 chunk pairs (one block -> two), 3 -> 6, 10 -> 15
    out = [hairpin_design(100 + n, n) for n in (30, 64, 65, 66, 85, 86, 129, 130, 257, 258)]
    out.append(coulomb_chain(seed=41, n=66, box=46.0))
    out.append(compact_allpairs(seed=42, ions=True, periodic=True))
    out.append(small_ions_box(seed=43))
    return out


def test_energies_at_the_edges_of_the_split():
    cases = _cases()
    eng = Engine([s for s, _ in cases], seed=3)
    for k, (_, x) in enumerate(cases):
        eng.set_coords(k, x)
    eng.neighbor(-1)
    eng.force_all()
    every = eng.energy_all()
    pick = [k for k in range(len(cases) - 1, -1, -2)] + [0, 0]
    some = eng.energy_systems(pick)
    for row, k in zip(some, pick):
        assert np.array_equal(row, every[k])
    for k, (s, x) in enumerate(cases):
        print(f"[energy parts] nt {s.nmp // 3 + 1} beads {s.nmp}", flush=True)
        assert np.array_equal(eng.energy_sumup(k), every[k])
        o = oracle.Oracle(s)
        o.neighbor(x)
        o.force(x, seed=3, sys_id=k, step=0)
        eo = np.asarray(o.energy(x, np.zeros_like(x)))
        # FP64 sums in another order, the contact coefficient from FP32
        # square roots of epsilon (6e-8 relative): 1e-7 of the largest term
        assert np.abs(every[k] - eo).max() <= 1e-7 * np.abs(eo[1:]).max()
    eng.close()
