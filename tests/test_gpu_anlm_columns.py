"""The column a_nlm kernel (matrix cores, a wave per neighbor species) and the
order-1/2 features it forms, against the CPU oracle and the register kernel at
the edges of its range: l_max 1 to 12 (below and at the 5, 9 and 13 steps of its
instances), 1 to 16 radial functions and 17 (the two-tile kernel), one and two
species, from no neighbors and ragged steps of four to several batches of 64.

Bars: a_nlm within 1e-13 of the largest (sums of up to ~300 terms of unit
roundoff 1.1e-16), energy 1e-10 eV/atom and forces 1e-8 of the largest."""
import numpy as np
import pytest

import oracle_lib as O
from common import rel_force_err
from mlip_hip import PairMLIPGtinv, inspect_model
from mlip_hip import workloads as W
from test_gpu_intermediates import device_anlm, oracle_anlm

pytestmark = pytest.mark.gpu


def potential(path, elements, maxl, nfn):
    def write(coeffs):
        W.write_potential(path, elements, 5.0, 2, 2, maxl, 3, [maxl, min(maxl, 2)], [0, 0], coeffs,
                          [(1.0, mu) for mu in np.linspace(0.0, 4.5, nfn)], [30.0] * len(elements))
    write([0.0])
    write(np.random.default_rng(maxl + nfn).normal(0.0, 1e-3, size=inspect_model(path, 4)))
    return path


@pytest.mark.parametrize("elements,maxl,nfn,natoms,density,rmin", [
    (("X",), 12, 16, 23, 0.35, 0.9), (("Ti", "Al"), 12, 12, 31, 0.55, 0.7), (("Ti", "Al"), 3, 16, 9, 0.1, 1.4),
    (("Ti", "Al"), 4, 1, 17, 0.05, 1.8), (("Ti", "Al"), 1, 5, 40, 0.27, 0.9), (("X",), 2, 4, 3, 0.02, 1.8),
    (("Ti", "Al"), 7, 13, 70, 0.03, 1.8), (("Ti", "Al"), 11, 3, 12, 0.06, 1.5), (("Ti", "Al"), 8, 8, 2, 0.002, 1.5),
    (("Ti", "Al"), 4, 17, 20, 0.06, 1.5)])
def test_against_oracle_and_register_kernel(tmp_path, elements, maxl, nfn, natoms, density, rmin):
    pot = potential(str(tmp_path / "p.mlip"), elements, maxl, nfn)
    s = W.random_cell_structure(natoms, density, np.random.default_rng(natoms), rmin=rmin,
                                type_fraction=0.4 if len(elements) == 2 else None)
    o = O.Oracle(pot)
    ro = o.compute(W.build_neighbor_list(s, o.cutoff), s.types - 1)
    ao = oracle_anlm(o, s, maxl)
    scale = np.abs(ao).max()
    p = PairMLIPGtinv()
    p.settings()
    p.coeff("*", "*", pot, *elements)
    nl = W.build_neighbor_list(s, p.init_one(), full=True)
    for kind in ("mfma", "registers"):
        p.set_anlm_kernel(kind)
        r = p.compute(nl, nl.types)
        a = device_anlm(p, s.types - 1)
        assert np.abs(a - ao).max() <= 1e-13 * scale, kind
        assert abs(r["energy"] - ro["energy"]) <= 1e-10 * natoms * max(1.0, abs(ro["energy"]) / natoms), kind
        if np.abs(ro["forces"]).max() > 0.0:
            assert rel_force_err(r["forces"], ro["forces"]) <= 1e-8, kind
