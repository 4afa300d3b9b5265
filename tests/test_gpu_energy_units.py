"""energy_unit of systems of many units: the parts of each unit pair's sums stay
bounded in number and memory, and the entries are the oracle's."""
import numpy as np
import pytest

import oracle
from tis_amd import topology as T
from tis_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("units,nt", [(5, 90), (20, 30), (60, 8)])
def test_energy_unit_of_many_units(units, nt):
    rng = np.random.default_rng(8)
    s = T.build_rna_system([(T.random_sequence(rng, nt), []) for _ in range(units)], name="units")
    x = T.compact_coords(s, rng, box=4.5 * s.nmp ** (1 / 3) + 10, min_dist=2.6)
    print(f"[energy units] {units} units {s.nmp} beads", flush=True)
    eng = Engine([s], keys=[0], seed=0)
    eng.set_coords(0, x)
    eng.neighbor(0)
    eng.force_sumup(0)
    o = oracle.Oracle(s)
    o.neighbor(x)
    o.force(x, seed=0, sys_id=0, step=0)
    before = eng.device_bytes()
    for style in (0, 1):
        eu, euo = eng.energy_unit(0, style), o.energy_unit(x, np.zeros_like(x), style)
        # FP64 sums in another order, the contact coefficient from FP32 square
        # roots of epsilon: 1e-7 of the entry, or of its type's largest
        top = np.abs(euo).max(axis=(0, 1), keepdims=True)
        assert (np.abs(eu - euo) <= 1e-7 * np.maximum(np.abs(euo), top)).all()
    # 25 entries a unit pair, 9 sums a part, 4,096 parts or one a pair
    nn = units * units
    assert eng.device_bytes() - before <= 8 * (25 * nn + 9 * max(nn, 4096))
    eng.close()
