"""The per-atom pass leaves the evaluation's adjoint weights H = lin + D W (models
without cubic terms) as they were: fetched after a call with per-atom outputs they
are the ones of a call without, bit for bit.  864 atoms take the small-tile product,
10,976 the tiled one."""
import numpy as np
import pytest

from common import config_potential
from mlip_hip import PairMLIPGtinv
from mlip_hip import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("edge", [6, 14])
def test_weights_kept(edge):
    p = PairMLIPGtinv()
    p.settings()
    p.coeff("*", "*", config_potential("binary_order4_quadratic"), "Ti", "Al")
    s = W.fcc(edge, 4.0, 0.08, 4, type_fraction=0.5, type_seed=4)
    nl = W.build_neighbor_list(s, p.init_one(), full=True)

    def weights(atomic):
        p.compute(nl, nl.types, eatom=atomic, vatom=atomic)
        lay = p.debug_fetch(6, 8).astype(int)
        assert lay[7] == 1
        n_pr, rows, out = lay[0], 0, []
        h = p.debug_fetch(4, 1 << 28)[:64 * (lay[3] + lay[6]) * n_pr].reshape(-1, n_pr)
        for t in range(2):  # a species' slots are its atoms, then the last block's empty ones
            n = int((s.types == t + 1).sum())
            out.append(h[rows:rows + n, :lay[2 + 3 * t]].copy())
            rows += 64 * lay[3 + 3 * t]
        return out

    for a, b in zip(weights(False), weights(True)):
        assert a.size and np.array_equal(a, b)
