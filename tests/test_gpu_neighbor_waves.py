"""The wave-per-atom list build where its parts change shape, bit for bit against
the host builder: more members in 64 stencil bins than one part of the LDS list
holds, stencils of fewer and more than 64 bins and not multiples of it, empty
bins, fewer atoms than waves in a workgroup, and no pairs at all."""
import numpy as np
import pytest

from common import config_potential
from mlip_hip import ResidentSystem, periodic_full_list
from mlip_hip import workloads as W
from test_gpu_neighbor import check_lists, gpu_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("natoms,lengths", [
    (1500, (13.0, 11.0, 12.5)), (300, (3.0, 4.0, 5.0)), (3, (2.0, 30.0, 5.0)), (2, (40.0, 40.0, 40.0)),
    (700, (60.0, 3.5, 3.5)), (5, (1.5, 1.6, 1.7))])
def test_lists_bit_exact(natoms, lengths):
    rng = np.random.default_rng(natoms)
    cell = np.diag(lengths)
    cell[1, 0], cell[2, 0], cell[2, 1] = 0.21 * lengths[0], -0.13 * lengths[0], 0.17 * lengths[1]
    pos = rng.uniform(-0.5, 1.5, size=(natoms, 3)) @ cell
    s = W.Structure(cell, pos, np.ones(natoms, dtype=np.int32))
    p = gpu_pair(config_potential("fcc256_order3_linear"), ["X"])
    rs = ResidentSystem.from_cell(p, s.cell, s.positions, s.types)
    off, idx, sh = periodic_full_list(s.cell, s.positions, p.init_one())
    check_lists(rs.lists(), off, idx, sh, (natoms, lengths))
