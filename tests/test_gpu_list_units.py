"""The list blocks (units of 32 beads or charges dealt out to a block's waves)
at the edges of units, tiles and rounds of 64 units against the oracle's
lists, and the launches of many tiles (fewer waves per block) against a system
alone, bit for bit."""
import numpy as np
import pytest

import oracle
from systems import coulomb_chain, hairpin_design
from tis_amd import topology as T
from tis_amd.engine import LIST_ELE, LIST_EXV, Engine

pytestmark = pytest.mark.gpu


def _sorted(p):
    return p[np.lexsort(p.T[::-1])]


@pytest.mark.parametrize("nt", [33, 43, 54, 64, 65, 107, 129, 690])
def test_lists_equal_the_oracle(nt):
    # 690 nt: 2,069 beads, 65 units
    s, x = coulomb_chain(seed=nt, n=nt, rcut=30.0, box=3.2 * nt ** 0.5 + 24.0) if nt < 200 else hairpin_design(nt, nt)
    print(f"[list units] nt={nt} beads={s.nmp}", flush=True)
    e = Engine([s])
    e.set_coords(0, x)
    e.neighbor(0)
    o = oracle.Oracle(s)
    o.neighbor(x)
    assert np.array_equal(_sorted(e.pairs(0, LIST_EXV)), _sorted(o.lists(0)))
    assert np.array_equal(_sorted(e.pairs(0, LIST_ELE)[0]), _sorted(o.lists(1)[0]))
    e.close()


def test_units_of_many_kinds_equal_the_oracle():
    """18 units: the radius table stays in memory."""
    rng = np.random.default_rng(8)
    s = T.build_rna_system([(T.random_sequence(rng, 8), []) for _ in range(18)], name="units18")
    x = T.compact_coords(s, rng, box=60, min_dist=2.6)
    e = Engine([s])
    e.set_coords(0, x)
    e.neighbor(0)
    o = oracle.Oracle(s)
    o.neighbor(x)
    assert np.array_equal(_sorted(e.pairs(0, LIST_EXV)), _sorted(o.lists(0)))
    e.close()


def test_many_tiles_equal_alone():
    base = [hairpin_design(300 + k, n) for k, n in enumerate([120, 97, 200])]
    n = 174   # 58 of each: 1,200 and more tiles
    batch = Engine([base[k % 3][0] for k in range(n)], keys=list(range(n)), seed=3)
    for k in range(n):
        batch.set_coords(k, base[k % 3][1])
    batch.neighbor(-1)
    fb = batch.force_all()
    for k in (0, 1, 2, n - 1):
        alone = Engine([base[k % 3][0]], keys=[k], seed=3)
        alone.set_coords(0, base[k % 3][1])
        alone.neighbor(0)
        assert np.array_equal(alone.force_sumup(0), fb[k])
        alone.close()
    batch.close()
