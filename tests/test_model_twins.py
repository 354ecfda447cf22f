"""Two order-2 families of one species pair and l: the model loads (the built-in table
has none, another may)."""
import os

import host_checks


def test_twin_families_load(tmp_path):
    table = os.path.join(os.path.dirname(host_checks.CSRC), "data", "gtinv_table.txt")
    host_checks.run(tmp_path, "twin_families", sources=["model.cpp"], args=[table, tmp_path])
