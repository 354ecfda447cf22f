"""mlip_compute_flat_noalloc accepts every structure whose buffers fit its 128 MiB
array with 7 x 128 doubles of reduction space: the largest number of dimers for
which they do is evaluated, and equals the allocating entry point bit for bit."""
import numpy as np
import pytest

from mlip_hip import PairMLIPGtinv, inspect_model
from mlip_hip import workloads as W

pytestmark = pytest.mark.gpu

SCRATCH = 128 << 20


def needed(n):
    """Bytes for n atoms with one neighbor each, a model of one species, one radial
    function, l_max 0 and no products: buffers at multiples of 256 bytes."""
    blocks = (n + 63) // 64
    slots = 64 * blocks
    lists = [24 * n, 4 * n, 4 * (n + 1), 4 * n, 4 * n, 4 * (n + 1), 8 * n]  # x, elements, pairs, gather lists
    layout = [4 * slots, 4 * n, 4 * blocks]
    work = [16 * slots, 16 * slots, 8, 8, 8, 8 * slots, 8 * slots, 96 * slots]  # a_nlm, G, products, energies
    out = [24 * n, 48 * n, 24 * n, 8 * slots, 8 * 7 * 128, 8 * 8]
    used = 0
    for b in lists + layout + work + out:
        used = (used + 255) // 256 * 256 + b
    return used


def test_largest_structure(tmp_path):
    path = str(tmp_path / "p.mlip")

    def write(coeffs):
        W.write_potential(path, ("X",), 5.0, 2, 1, 0, 2, [0], [0], coeffs, [(1.0, 2.0)], [30.0])
    write([0.0])
    write(np.linspace(0.1, 0.2, inspect_model(path, 4)))
    lo, hi = 2, SCRATCH // 256
    while hi - lo > 2:
        mid = (lo + hi) // 4 * 2
        lo, hi = (mid, hi) if needed(mid) <= SCRATCH else (lo, mid)
    n = lo
    assert needed(n) <= SCRATCH < needed(n + 2)
    k = np.arange(n)
    x = np.zeros((n, 3))
    x[:, 0] = 10.0 * (k // 2 % 500) + (k % 2) * np.random.default_rng(5).uniform(1.5, 3.0, size=n)
    x[:, 1] = 10.0 * (k // 1000)
    nl = W.NeighborList(x, (k + 1).astype(np.int64), np.ones(n, dtype=np.int32), n, k.astype(np.int32),
                        np.ones(n, dtype=np.int32), np.arange(n + 1, dtype=np.int32), (k ^ 1).astype(np.int32), True)
    p = PairMLIPGtinv()
    p.settings()
    p.coeff("*", "*", path, "X")
    b = p.compute(nl, nl.types, noalloc=True)
    a = p.compute(nl, nl.types)
    assert a["energy"] == b["energy"] != 0.0
    assert np.array_equal(a["virial"], b["virial"]) and np.array_equal(a["forces_all"], b["forces_all"])
    # the totals, over all energy and virial parts: dimers along x, each pair's virial
    # its separation times its force; n roundings at most
    f = a["forces_all"]
    want = ((x[1::2] - x[::2])[:, 0] * f[1::2, 0]).sum()
    assert abs(a["virial"][0] - want) <= n * 2.0 ** -53 * np.abs((x[1::2] - x[::2])[:, 0] * f[1::2, 0]).sum()
