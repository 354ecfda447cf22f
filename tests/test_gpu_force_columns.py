"""The matrix-core force kernel against the CPU oracle at the edges of its shape:
l_max below and at the 5, 9 and 13 levels of its instances, 1 to 16 radial
functions (one to four steps of four), one and two species, a species with no
neighbor, neighbor counts around tiles of 16 and beyond a batch of 176, and each
number of waves, which must not change a bit of the forces.

Bars: FP64 1e-8 of the largest force and virial component.  Mixed: each pair
force sums about 12 x 91 products rounded to FP32 (6e-8, near 1e-6 of its largest
term together), and the pair forces of a centre cancel by up to a hundred: 1e-4
of the largest."""
import numpy as np
import pytest

import oracle_lib as O
from mlip_hip import PairMLIPGtinv
from mlip_hip import workloads as W
from test_gpu_anlm_columns import potential

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("elements,maxl,nfn,natoms,density,rmin,fraction", [
    (("X",), 12, 16, 19, 0.4, 0.9, None), (("Ti", "Al"), 12, 12, 37, 0.42, 0.8, 0.5), (("Ti", "Al"), 8, 5, 24, 0.05, 1.6, 0.1),
    (("Ti", "Al"), 9, 8, 20, 0.06, 1.6, 0.0), (("Ti", "Al"), 4, 4, 30, 0.06, 1.6, 1.0), (("X",), 5, 9, 11, 0.03, 1.8, None),
    (("Ti", "Al"), 1, 1, 6, 0.03, 1.8, 0.5), (("Ti", "Al"), 3, 13, 2, 0.004, 1.8, 0.5)])
def test_against_oracle(tmp_path, elements, maxl, nfn, natoms, density, rmin, fraction):
    pot = potential(str(tmp_path / "p.mlip"), elements, maxl, nfn)
    s = W.random_cell_structure(natoms, density, np.random.default_rng(natoms), rmin=rmin, type_fraction=fraction)
    o = O.Oracle(pot)
    ro = o.compute(W.build_neighbor_list(s, o.cutoff), s.types - 1)
    fmax, vmax = np.abs(ro["forces"]).max(), np.abs(ro["virial"]).max()
    p = PairMLIPGtinv()
    p.settings()
    p.coeff("*", "*", pot, *elements)
    nl = W.build_neighbor_list(s, p.init_one(), full=True)
    for precision, tol in (("fp64", 1e-8), ("mixed", 1e-4)):
        p.set_precision(precision)
        first = None
        for threads in (256, 192, 128, 64):
            assert p.lib.mlip_set_force_threads(p.ctx, threads) == 0
            r = p.compute(nl, nl.types)
            f = r["forces"]
            assert np.abs(f - ro["forces"]).max() <= tol * fmax, (precision, threads)
            assert np.abs(r["virial"] - ro["virial"]).max() <= tol * vmax, (precision, threads)
            assert first is None or np.array_equal(f, first), (precision, threads)
            first = f
