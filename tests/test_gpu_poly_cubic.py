"""The cubic polynomial's kernel (a workgroup per slot, sixteen lanes per feature)
against the CPU oracle: fewer features than lane groups, more, term lists shorter
and longer than the lanes, one and two species (a species' empty slots).

Bars: the suite's FP64 ones (1e-10 eV/atom, 1e-8 of the largest component)."""
import numpy as np
import pytest

import oracle_lib as O
from common import rel_force_err
from mlip_hip import PairMLIPGtinv, inspect_model
from mlip_hip import workloads as W

pytestmark = pytest.mark.gpu


def potential(path, elements, maxl, nfn):
    def write(coeffs):
        W.write_potential(path, elements, 5.0, 2, 3, maxl, 2, [maxl], [0], coeffs,
                          [(1.0, mu) for mu in np.linspace(0.0, 4.0, nfn)], [30.0] * len(elements))
    write([0.0])
    write(np.random.default_rng(maxl + nfn).normal(0.0, 1e-3, size=inspect_model(path, 4)))
    return path


@pytest.mark.parametrize("elements,maxl,nfn,natoms", [
    (("X",), 0, 1, 3), (("X",), 2, 7, 65), (("Ti", "Al"), 1, 4, 33), (("Ti", "Al"), 2, 3, 5)])
def test_against_oracle(tmp_path, elements, maxl, nfn, natoms):
    pot = potential(str(tmp_path / "p.mlip"), elements, maxl, nfn)
    s = W.random_cell_structure(natoms, 0.05, np.random.default_rng(natoms), rmin=1.8,
                                type_fraction=0.4 if len(elements) == 2 else None)
    o = O.Oracle(pot)
    ro = o.compute(W.build_neighbor_list(s, o.cutoff), s.types - 1)
    p = PairMLIPGtinv()
    p.settings()
    p.coeff("*", "*", pot, *elements)
    nl = W.build_neighbor_list(s, p.init_one(), full=True)
    r = p.compute(nl, nl.types)
    assert abs(r["energy"] - ro["energy"]) <= 1e-10 * natoms * max(1.0, abs(ro["energy"]) / natoms)
    assert np.abs(r["virial"] - ro["virial"]).max() <= 1e-8 * np.abs(ro["virial"]).max()
    assert rel_force_err(r["forces"], ro["forces"]) <= 1e-8
