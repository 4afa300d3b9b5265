"""Periodic chunk pairs (a block each, a quarter of the steps per wave) and the
reciprocal pass (half of the vectors, quarters of the charge chunks) at the
edges of their tiles, with the lists
of such systems, every electrostatic form, against the FP64 oracle."""
import numpy as np
import pytest

import oracle
from systems import force_error
from tis_amd import topology as T
from tis_amd.engine import LIST_ELE, LIST_EXV, Engine
from tis_amd.sysdesc import ELE_COULOMB, ELE_DH, ELE_EWALD

pytestmark = pytest.mark.gpu


def _box(nq, form, hmax):
    """A 12-nt chain and as many ions as make nq charges, in a 60 A cube."""
    chain = int((np.abs(T.config2_ewald(5, n=12, box=60.0, n_mg=1, n_k=0, n_cl=0, rcut=25.0)[0].charge) > 1e-6).sum()) - 1
    ions = nq - chain
    s, x = T.config2_ewald(5, n=12, box=60.0, n_mg=0, n_k=ions // 2, n_cl=ions - ions // 2, alpha=0.2, rcut=25.0,
                           hmax=hmax)
    assert (np.abs(s.charge) > 1e-6).sum() == nq
    if form != ELE_EWALD:
        s2 = T.build_rna_system([(T.random_sequence(np.random.default_rng(5), 12), [])],
                                ions=["K"] * (ions // 2) + ["Cl"] * (ions - ions // 2), box=(60.0, 60.0, 60.0),
                                ele_form=form, cutoff_ele=2.0 if form == ELE_DH else 25.0, phos_charge=-1.0)
        return s2, x
    return s, x


@pytest.mark.parametrize("nq,form,hmax", [(16, ELE_EWALD, 1), (63, ELE_EWALD, 2), (64, ELE_EWALD, 4),
                                          (65, ELE_EWALD, 5), (127, ELE_COULOMB, 0), (128, ELE_DH, 0),
                                          (129, ELE_EWALD, 7), (193, ELE_EWALD, 3), (65, ELE_DH, 0),
                                          (193, ELE_COULOMB, 0)])
def test_forces_and_energies(nq, form, hmax):
    s, x = _box(nq, form, hmax)
    print(f"[periodic pairs] nq={nq} form={form} hmax={hmax}", flush=True)
    e = Engine([s], keys=[0], seed=0)
    e.set_coords(0, x)
    e.neighbor(0)
    f = e.force_sumup(0)
    en = e.energy_sumup(0)
    o = oracle.Oracle(s)
    o.neighbor(x)
    for which, k in ((LIST_EXV, 0), (LIST_ELE, 1)):
        a, b = e.pairs(0, which), o.lists(k)
        (a, ac), (b, bc) = (a, b) if k else ((a, np.zeros(len(a))), (b, np.zeros(len(b))))
        p, q = np.lexsort(a.T[::-1]), np.lexsort(b.T[::-1])
        assert np.array_equal(a[p], b[q]) and np.array_equal(ac[p], bc[q])
    fo, _ = o.force(x, seed=0, sys_id=0, step=0)
    eo = o.energy(x, np.zeros_like(x))
    err = force_error(f, fo).max()
    print("   force", err, flush=True)
    assert err <= 1e-5
    assert (np.abs(en - eo) / np.maximum(np.abs(eo), 1e-6)).max() <= 1e-7
    e.close()
