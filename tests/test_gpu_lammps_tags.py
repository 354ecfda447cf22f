"""Half neighbor lists whose tags are dense (a table finds a ghost's owner) and
sparse, huge or negative (a map does): the same results bit for bit, and a tag
with no local atom is refused by both."""
import numpy as np
import pytest

from common import config_potential
from mlip_hip import MlipError, PairMLIPGtinv
from mlip_hip import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natoms", [1, 7, 60])
def test_tag_forms_agree(natoms):
    s = W.random_cell_structure(natoms, 0.05, np.random.default_rng(natoms), rmin=1.8)
    p = PairMLIPGtinv()
    p.settings()
    p.coeff("*", "*", config_potential("fcc256_order3_linear"), "X")
    nl = W.build_neighbor_list(s, p.init_one(), full=False)
    base = p.compute(nl, nl.types)
    dense = nl.tag.copy()
    for form in (lambda t: 10**12 * t, lambda t: -t, lambda t: t + 3 * natoms, lambda t: t + 4 * natoms + 1100):
        nl.tag = form(dense.astype(np.int64))
        r = p.compute(nl, nl.types)
        assert r["energy"] == base["energy"]
        assert np.array_equal(r["forces_all"], base["forces_all"])
        assert np.array_equal(r["virial"], base["virial"])
        used = nl.idx[nl.idx >= natoms]
        if used.size:
            nl.tag[used[0]] = 10**15 + 1
            with pytest.raises(MlipError, match="local owner"):
                p.compute(nl, nl.types)
