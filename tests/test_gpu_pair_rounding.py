"""Rounding of the radial style's polynomial step.  The products of pair-60 reach 1e5
against energies of a few eV, so the order in which they are added decides how much
of the result is lost.  The engine's forces are compared with 80-bit ones on the
same pair vectors; their rms error may be no larger than that of the plain method:
every feature's sum, and every derivative's sum over its terms, as one FP64 chain in
the coefficients' order."""
import numpy as np
import pytest

from common import ref
from mlip_hip import PairMLIPGtinv, inspect_model
from mlip_hip import workloads as W

pytestmark = pytest.mark.gpu


def read_pair_potential(path):
    lines = open(path).read().splitlines()
    n = int(lines[7].split()[0])
    w = np.array(lines[8].split()[:n], dtype=float) / np.array(lines[9].split()[:n], dtype=float)
    nfn = int(lines[10].split()[0])
    beta, mu = np.array([lines[11 + k].split()[:2] for k in range(nfn)], dtype=float).T
    return float(lines[1].split()[0]), w, beta, mu


def forces(pot, nl, two, three, real):
    """Forces in the number type `real`, all sums as chains."""
    rc, w, beta, mu = pot
    nfn, cen = len(mu), np.repeat(nl.ilist, np.diff(nl.off))
    d = (nl.x[cen] - nl.x[nl.idx])  # FP64 in any case: the engine's pair vectors
    keep = np.sqrt((d * d).sum(1)) < rc
    cen, nbr, d = cen[keep], np.asarray(nl.idx)[keep], d[keep].astype(real)
    r = np.sqrt((d * d).sum(1))
    k = real(3.141592653589793) / real(rc)
    fc, fd = (np.cos(k * r) + 1) / 2, -k / 2 * np.sin(k * r)
    t = r[:, None] - mu.astype(real)
    g = np.exp(-beta.astype(real) * t * t)
    # type combination of (centre, neighbor): 0-0, 0-1, 1-1
    feat = (nl.types[cen] - 1 + nl.types[nbr] - 1)[:, None] * nfn + np.arange(nfn)
    D = np.zeros((nl.nlocal, 3 * nfn), dtype=real)
    np.add.at(D, (cen[:, None], feat), g * fc[:, None])
    H = np.zeros_like(D)
    n_des, wr = 3 * nfn, w.astype(real)
    for m, (a, b) in enumerate(two):
        H[:, a] += wr[n_des + m] * D[:, b]
        H[:, b] += wr[n_des + m] * D[:, a]
    for m, (a, b, c) in enumerate(three):
        q = wr[n_des + len(two) + m]
        H[:, a] += q * (D[:, b] * D[:, c])
        H[:, b] += q * (D[:, a] * D[:, c])
        H[:, c] += q * (D[:, a] * D[:, b])
    H += wr[:n_des]
    de = (g * (fd[:, None] - 2 * beta.astype(real) * t * fc[:, None]) * H[cen[:, None], feat]).sum(1)
    f = np.zeros((len(nl.x), 3), dtype=real)
    pf = (de / r)[:, None] * d
    np.add.at(f, cen, -pf)
    np.add.at(f, nbr, pf)
    out = np.zeros((nl.nlocal, 3), dtype=real)
    np.add.at(out, nl.owner, f)
    return out


def test_force_error_not_above_a_chain():
    path = ref("pair-60.mlip")
    pot, two, three = read_pair_potential(path), inspect_model(path, 2), inspect_model(path, 3).reshape(-1, 3)
    p = PairMLIPGtinv()
    p.settings()
    p.coeff("*", "*", path, "Ti", "Al")
    for seed in (1, 2):
        s = W.fcc(4, 4.05, 0.08, seed, type_fraction=0.5, type_seed=seed)
        nl = W.build_neighbor_list(s, p.init_one(), full=True)
        exact = forces(pot, nl, two, three, np.longdouble)
        rms = lambda v: float(np.sqrt((v * v).mean()))  # noqa: E731
        chain = rms(forces(pot, nl, two, three, np.float64) - exact) / rms(exact)
        here = rms(p.compute(nl, nl.types)["forces"] - exact) / rms(exact)
        print("rms force error: here %.2e, one chain %.2e" % (here, chain), flush=True)
        assert here <= chain
