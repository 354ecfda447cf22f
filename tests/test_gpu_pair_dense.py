"""Radial-only style on the dense derivative product (k_pair_poly_dense) and on
the derivative lists: energy, forces, virial and the per-atom split against the
CPU oracle, over one and two species, every max_p, radial counts on both sides
of the 8 / 16 / 32-wide sums and of the 16-column tiles, and atom counts at the
edges of a 16-centre tile and of a 64-slot block.

Bars: the suite's FP64 ones (1e-10 eV/atom, 1e-8 of the largest component)."""
import numpy as np
import pytest

import oracle_lib as O
from common import rel_force_err
from mlip_hip import PairMLIPGtinv, inspect_model
from mlip_hip import workloads as W

pytestmark = pytest.mark.gpu


def potential(path, elements, model_type, maxp, nfn):
    def write(coeffs):
        with open(path, "w") as fh:
            fh.write("%s # element\n5.0 # cutoff\ngaussian # pair_type\npair # des_type\n" % " ".join(elements))
            fh.write("%d # model_type\n%d # max_p\n0 # max_l\n%d # n\n" % (model_type, maxp, len(coeffs)))
            fh.write(" ".join("%.17g" % v for v in coeffs) + "\n")
            fh.write(" ".join("1.0" for _ in coeffs) + "\n%d # number of parameters\n" % nfn)
            for mu in np.linspace(0.0, 4.5, nfn):
                fh.write("1.0 %.17g # pair func. params\n" % mu)
            fh.write(" ".join("30.0" for _ in elements) + " # atomic mass\n")
    write([0.0])
    n = inspect_model(path, 4)
    write(np.random.default_rng(nfn + 10 * maxp).normal(0.0, 1e-3, size=n))
    return path


@pytest.mark.parametrize("elements,model_type,maxp,nfn,natoms",
                         [(("X",), 2, 2, 3, 1), (("X",), 2, 3, 9, 15), (("Ti", "Al"), 2, 3, 8, 65),
                          (("Ti", "Al"), 2, 2, 17, 33), (("Ti", "Al"), 2, 3, 32, 17), (("Ti", "Al"), 1, 3, 16, 31),
                          (("Ti", "Al"), 2, 1, 5, 16)])
def test_dense_and_list_forms(tmp_path, elements, model_type, maxp, nfn, natoms):
    pot = potential(str(tmp_path / "p.mlip"), elements, model_type, maxp, nfn)
    s = W.random_cell_structure(natoms, 0.05, np.random.default_rng(natoms), rmin=1.8,
                                type_fraction=0.5 if len(elements) == 2 else None)
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

    assert abs(r["energy"] - ro["energy"]) <= 1e-10 * natoms
    assert np.abs(r["virial"] - ro["virial"]).max() <= 1e-8 * np.abs(ro["virial"]).max()
    if natoms > 1:
        assert rel_force_err(r["forces"], ro["forces"]) <= 1e-8
    assert np.abs(fold(nl, r["eatom"]) - fold(nl_o, ro["eatom"])).max() <= 1e-10
    va = fold(nl_o, ro["vatom"])
    assert np.abs(fold(nl, r["vatom"]) - va).max() <= 1e-8 * np.abs(va).max()
