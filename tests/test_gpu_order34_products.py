"""Order-3 and order-4 adjoint kernels that form each product once (k_q3, k_q4)
and the rows of order 1/2 they carry, against the CPU oracle where their tables
change shape: one and two species, order-3 l from 0 to 10 (five and six rows per
segment, divided segments), l_max below, at and above the tile and the
12-level limit, order-4 l of 0..2, and families in the polynomial, which the
order-3/4 kernel keeps.  Per-atom energy and virial check the split weights.

Bars: the suite's FP64 ones (1e-10 eV/atom, 1e-8 of the largest component)."""
import numpy as np
import pytest

import oracle_lib as O
from common import rel_force_err
from mlip_hip import PairMLIPGtinv, inspect_model
from mlip_hip import workloads as W

pytestmark = pytest.mark.gpu


def potential(path, elements, model_type, maxp, maxl, gtinv_maxl, nfn):
    def write(coeffs):
        W.write_potential(path, elements, 5.0, model_type, maxp, maxl, len(gtinv_maxl) + 1, gtinv_maxl,
                          [0] * len(gtinv_maxl), coeffs, [(1.0, mu) for mu in np.linspace(0.0, 4.0, nfn)],
                          [30.0] * len(elements))
    write([0.0])
    write(np.random.default_rng(maxl + nfn).normal(0.0, 1e-2, size=inspect_model(path, 4)))
    return path


@pytest.mark.parametrize("elements,model_type,maxp,maxl,gtinv_maxl,nfn,natoms", [
    (("X",), 2, 1, 4, [4, 4, 2], 3, 5), (("X",), 4, 2, 10, [10, 10], 2, 33),
    (("Ti", "Al"), 2, 2, 2, [2, 2, 2], 1, 17), (("Ti", "Al"), 4, 2, 6, [6, 5, 1], 3, 70),
    (("Ti", "Al"), 3, 2, 12, [12, 9], 2, 9), (("Ti", "Al"), 2, 1, 1, [1, 1, 1], 2, 3),
    (("Ti", "Al"), 4, 2, 14, [14, 3, 2], 2, 20), (("Ti", "Al"), 4, 1, 2, [2, 0, 2], 2, 12),
    (("Ti", "Al"), 2, 1, 8, [3, 8, 2], 1, 1)])
def test_against_oracle(tmp_path, elements, model_type, maxp, maxl, gtinv_maxl, nfn, natoms):
    pot = potential(str(tmp_path / "p.mlip"), elements, model_type, maxp, maxl, gtinv_maxl, nfn)
    s = W.random_cell_structure(natoms, 0.05, np.random.default_rng(natoms), rmin=1.8,
                                type_fraction=0.4 if len(elements) == 2 else None)
    o = O.Oracle(pot)
    nl_o = W.build_neighbor_list(s, o.cutoff, full=False)
    ro = o.compute(nl_o, s.types - 1, eatom=True, vatom=True)
    p = PairMLIPGtinv()
    p.settings()
    p.coeff("*", "*", pot, *elements)
    nl = W.build_neighbor_list(s, p.init_one(), full=True)
    r = p.compute(nl, nl.types, eatom=True, vatom=True)

    def fold(lst, v):
        out = np.zeros((s.natoms,) + v.shape[1:])
        np.add.at(out, lst.owner, v)
        return out

    escale = max(1.0, abs(ro["energy"]) / natoms)
    assert abs(r["energy"] - ro["energy"]) <= 1e-10 * natoms * escale
    assert np.abs(r["virial"] - ro["virial"]).max() <= 1e-8 * np.abs(ro["virial"]).max()
    if natoms > 1:
        assert rel_force_err(r["forces"], ro["forces"]) <= 1e-8
    assert np.abs(fold(nl, r["eatom"]) - fold(nl_o, ro["eatom"])).max() <= 1e-10 * escale
    va = fold(nl_o, ro["vatom"])
    assert np.abs(fold(nl, r["vatom"]) - va).max() <= 1e-8 * np.abs(va).max()
