"""Merged rows of the linear order-5/6 families (k_qhigh_rows): per-atom
energy and virial (the rows scaled by 1 / order) and forces against the CPU
oracle at the edges of a slot block (one centre, 63, 65 of a species) and on
the all-families linear model, where both orders add to the same adjoint rows.

Bars: the suite's FP64 ones, 1e-10 eV/atom for energies and 1e-8 of the
largest component for forces and virials (rounding is six orders below)."""
import numpy as np
import pytest

import oracle_lib as O
from common import config_potential, rel_force_err
from mlip_hip import PairMLIPGtinv
from mlip_hip import workloads as W

pytestmark = pytest.mark.gpu


def cell(natoms):
    """natoms random positions at least 2.2 A apart, species at random."""
    return W.random_cell_structure(natoms, 0.03, np.random.default_rng(natoms), rmin=2.2, type_fraction=0.5)


@pytest.mark.parametrize("natoms", [1, 2, 63, 130])
def test_split_and_forces(natoms):
    name = "binary_order6_l20_linear"
    o = O.Oracle(config_potential(name))
    s = cell(natoms)
    nl_o = W.build_neighbor_list(s, o.cutoff, full=False)
    ro = o.compute(nl_o, s.types - 1, eatom=True, vatom=True)
    p = PairMLIPGtinv()
    p.settings()
    p.coeff("*", "*", config_potential(name), "Ti", "Al")
    nl = W.build_neighbor_list(s, p.init_one(), full=True)
    r = p.compute(nl, nl.types, eatom=True, vatom=True)

    def fold(lst, v):
        out = np.zeros((s.natoms,) + v.shape[1:])
        np.add.at(out, lst.owner, v)
        return out

    assert abs(r["energy"] - ro["energy"]) <= 1e-10 * natoms
    assert np.abs(r["virial"] - ro["virial"]).max() <= 1e-8 * np.abs(ro["virial"]).max()
    if natoms > 1:
        assert rel_force_err(r["forces"], ro["forces"]) <= 1e-8
    assert np.abs(fold(nl, r["eatom"]) - fold(nl_o, ro["eatom"])).max() <= 1e-10
    va = fold(nl_o, ro["vatom"])
    assert np.abs(fold(nl, r["vatom"]) - va).max() <= 1e-8 * np.abs(va).max()
