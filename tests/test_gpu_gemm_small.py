"""The few-row quadratic-form kernel (k_gemm_small): against numpy like the tiled
kernel, on forms whose width is not a multiple of its 16, 64 and 128-wide tiles
and rounds, and bit for bit equal to the tiled kernel's rows (a structure alone,
few rows, and inside a batch large enough for the tiled kernel).

Bar of test_gpu_gemm: 1e-13 of the term scale."""
import numpy as np
import pytest

from common import config_potential
from mlip_hip import BatchSystem, PairMLIPGtinv, inspect_model
from mlip_hip import workloads as W
from test_gpu_gemm import check_forms

pytestmark = pytest.mark.gpu


def pair(pot, elements=("Ti", "Al")):
    p = PairMLIPGtinv()
    p.settings()
    p.coeff("*", "*", pot, *elements)
    return p


@pytest.mark.parametrize("elements,maxl,nfn,natoms", [(("X",), 2, 3, 5), (("Ti", "Al"), 3, 5, 70),
                                                      (("Ti", "Al"), 6, 7, 33), (("X",), 12, 16, 20)])
def test_form_widths(tmp_path, elements, maxl, nfn, natoms):
    pot = str(tmp_path / "p.mlip")

    def write(coeffs):
        W.write_potential(pot, elements, 5.0, 4, 2, maxl, 2, [maxl], [0], coeffs,
                          [(1.0, mu) for mu in np.linspace(0.0, 4.0, nfn)], [30.0] * len(elements))
    write([0.0])
    write(np.random.default_rng(nfn).normal(0.0, 1e-2, size=inspect_model(pot, 4)))
    s = W.random_cell_structure(natoms, 0.05, np.random.default_rng(natoms), rmin=1.8,
                                type_fraction=0.4 if len(elements) == 2 else None)
    p = pair(pot, elements)
    nl = W.build_neighbor_list(s, p.init_one(), full=True)
    p.compute(nl, nl.types)
    lay = p.debug_fetch(6, 8)
    print("widths", int(lay[2]), int(lay[5]))
    check_forms(p, "maxl %d nfn %d" % (maxl, nfn), fused=1)


def test_rows_equal_in_either_kernel():
    pot = config_potential("binary_order4_quadratic")
    structs = W.random_structures(48, 64, 256, seed=11)
    big = BatchSystem(pair(pot), structs)
    big.compute()
    r = big.get()
    for k in (0, 17, 47):
        one = BatchSystem(pair(pot), [structs[k]])
        one.compute()
        a = one.get()
        assert a["energies"][0] == r["energies"][k]
        assert np.array_equal(a["forces"][0], r["forces"][k])
        assert np.array_equal(a["virials"][0], r["virials"][k])
