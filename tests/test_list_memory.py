"""The host memory that a context keeps between LAMMPS calls follows the calls, and a
context that goes on with a resident structure, a batch or a pool gives it back."""
import ctypes

import numpy as np
import pytest

import host_checks
from common import ref
from mlip_hip import BatchSystem, PairMLIPGtinv, RequestPool, ResidentSystem
from mlip_hip import workloads as W


def test_kept_lists_follow_the_calls(tmp_path):
    host_checks.run(tmp_path, "lists_kept")


class _MallInfo(ctypes.Structure):
    _fields_ = [(k, ctypes.c_size_t) for k in ("arena", "ordblks", "smblks", "hblks", "hblkhd", "usmblks", "fsmblks",
                                               "uordblks", "fordblks", "keepcost")]


def allocated_bytes():
    """Bytes of the C library's heap in use (freed ones may stay in the process)."""
    f = ctypes.CDLL(None).mallinfo2
    f.restype = _MallInfo
    m = f()
    return m.uordblks + m.hblkhd


@pytest.mark.gpu
@pytest.mark.parametrize("then", ["smaller call", "resident", "batch", "pool"])
def test_memory_given_back(then):
    # 12 million directed pairs (all but a few beyond the cutoff): 192 MB of lists
    n, per = 60000, 200
    k = np.arange(n, dtype=np.int32)
    x = np.zeros((n, 3))
    x[:, 0], x[:, 1] = 3.0 * (k % 300), 3.0 * (k // 300)
    idx = ((k[:, None] + 1 + np.arange(per)) % n).astype(np.int32).ravel()
    nl = W.NeighborList(x, k.astype(np.int64) + 1, np.ones(n, dtype=np.int32), n, k, np.full(n, per, dtype=np.int32),
                        (per * np.arange(n + 1)).astype(np.int32), idx, True)
    p = PairMLIPGtinv()
    p.settings()
    p.coeff("*", "*", ref("pair-17.mlip"), "Ti", "Al")
    s = W.fcc(2, 4.05, 0.05, 1, type_fraction=0.5, type_seed=1)
    small = W.build_neighbor_list(s, p.init_one(), full=True)
    p.compute(small, small.types)
    p.compute(nl, nl.types)
    before = allocated_bytes()
    if then == "smaller call":
        p.compute(small, small.types)
    elif then == "resident":
        ResidentSystem.from_cell(p, s.cell, s.positions, s.types).compute()
    elif then == "batch":
        BatchSystem(p, [s]).compute()
    else:
        RequestPool(p, 256, 65536, 1)
    given = before - allocated_bytes()
    print("%s: %.0f MB given back" % (then, given / 1e6), flush=True)
    assert given >= 100e6
