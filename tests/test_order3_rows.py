"""The order-3 kernel's rows above its tile: every read within its row for all
order-3 l (0..10) and l_max (to 20), and on the device, where the rows above a
short tile are fewer than the waves that take them, against the CPU oracle.

Bars: the suite's FP64 ones (1e-10 eV/atom, 1e-8 of the largest component)."""
import numpy as np
import pytest

import host_checks
import oracle_lib as O
from common import rel_force_err
from mlip_hip import PairMLIPGtinv, inspect_model
from mlip_hip import workloads as W


def test_row_walk_stays_in_its_rows(tmp_path):
    host_checks.run(tmp_path, "q3_rows")


@pytest.mark.gpu
@pytest.mark.parametrize("lmaxq3,maxl", [(0, 1), (0, 2), (0, 3), (1, 2), (2, 3), (2, 4)])
def test_short_rows_against_oracle(tmp_path, lmaxq3, maxl):
    path, elements, natoms = str(tmp_path / "p.mlip"), ("Ti", "Al"), 11

    def write(coeffs):
        W.write_potential(path, elements, 5.0, 4, 1, maxl, 3, [maxl, lmaxq3], [0, 0], coeffs,
                          [(1.0, mu) for mu in (0.0, 2.0, 4.0)], [30.0, 30.0])
    write([0.0])
    write(np.random.default_rng(maxl).normal(0.0, 1e-2, size=inspect_model(path, 4)))
    s = W.random_cell_structure(natoms, 0.05, np.random.default_rng(natoms), rmin=1.8, type_fraction=0.4)
    o = O.Oracle(path)
    ro = o.compute(W.build_neighbor_list(s, o.cutoff, full=False), s.types - 1)
    p = PairMLIPGtinv()
    p.settings()
    p.coeff("*", "*", path, *elements)
    nl = W.build_neighbor_list(s, p.init_one(), full=True)
    r = p.compute(nl, nl.types)
    assert abs(r["energy"] - ro["energy"]) <= 1e-10 * natoms * max(1.0, abs(ro["energy"]) / natoms)
    assert rel_force_err(r["forces"], ro["forces"]) <= 1e-8
    assert np.abs(r["virial"] - ro["virial"]).max() <= 1e-8 * np.abs(ro["virial"]).max()
