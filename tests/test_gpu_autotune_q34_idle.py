"""The order-3/4 plan of a model that gives the order-3/4 kernel no visits is kept:
no candidate is timed.  A model with order-3 families in the polynomial takes one of
the candidates."""
import pytest

from common import config_potential, ref
from mlip_hip import PairMLIPGtinv, ResidentSystem
from mlip_hip import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pot,kept", [("binary_order4_quadratic", True), ("gtinv-197.mlip", False)])
def test_plan_without_visits_is_kept(pot, kept):
    p = PairMLIPGtinv()
    p.settings()
    p.coeff("*", "*", ref(pot) if pot.endswith(".mlip") else config_potential(pot), "Ti", "Al")
    s = W.fcc(3, 4.05, 0.05, 1, type_fraction=0.5, type_seed=1)
    rs = ResidentSystem.from_cell(p, s.cell, s.positions, s.types)
    rs.compute()
    e = rs.get()["energy"]
    mine = (5, 77, 3)  # no candidate
    rs.set_q34_plan(*mine)
    assert (tuple(rs.autotune_q34(reps=1)) == mine) == kept
    rs.compute()
    assert abs(rs.get()["energy"] - e) <= 1e-10 * s.natoms
