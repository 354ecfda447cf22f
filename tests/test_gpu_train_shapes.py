"""Training outputs at the launch shapes of the feature-derivative kernel
(features and pairs per workgroup shrink as l_max grows; 16-feature and 4-pair
tiles) against the CPU oracle: l_max 8 and 12, one and two species, atom counts
1, 2 and 5 and pair counts that do not divide by the tiles.

Bars as in test_gpu_train.compare."""
import numpy as np
import pytest

import oracle_lib as O
from common import config_potential
from mlip_hip import PairMLIPGtinv, ResidentSystem
from mlip_hip import workloads as W
from test_gpu_train import compare

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,natoms", [("fcc256_order3_linear", 1), ("fcc256_order3_linear", 5),
                                         ("binary_order3_l10", 2)])
def test_shapes(name, natoms):
    elements = W.CONFIG_MODELS[name]["elements"]
    s = W.random_cell_structure(natoms, 0.02, np.random.default_rng(natoms), rmin=2.0,
                                type_fraction=0.5 if len(elements) == 2 else None)
    pot = config_potential(name)
    o = O.Oracle(pot)
    ro = o.train(W.build_neighbor_list(s, o.cutoff, full=False), s.types - 1)
    p = PairMLIPGtinv()
    p.settings()
    p.coeff("*", "*", pot, *elements)
    r = ResidentSystem.from_cell(p, s.cell, s.positions, s.types).train_features()
    compare({k: (r[k][0] if k == "SF" else r[k]) for k in r}, ro, "%s %d" % (name, natoms))
