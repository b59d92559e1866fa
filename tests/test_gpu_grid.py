"""Grid set-up on the device: the order of the points is that of a recursive bisection, points and weights are
the FP64 oracle's."""
import numpy as np
import pytest

import chinium_amd as ca
import oracle_lib as ol
from chinium_amd import workloads as wl

pytestmark = pytest.mark.gpu
CORE = 0.3  # bohr: points this close to a nucleus with Z > 2 are batched per atom


def _check_split(P):
    """P is a recursive bisection's order: its first 64 * (batches // 2) points lie on the lower side of the
    longest axis of the bounding box, and both parts are the same in themselves."""
    n = len(P)
    if n <= 64:
        return
    ax = int(np.argmax(P.max(0) - P.min(0)))  # the first of equal ones
    left = 64 * (((n + 63) // 64) // 2)
    assert P[:left, ax].max() <= P[left:, ax].min()
    _check_split(P[:left])
    _check_split(P[left:])


def _molecule(name):
    if name == "h2o":
        Z, X = wl.water_monomer_angstrom()
    elif name == "water9":
        Z, X = wl.water_cluster_angstrom(9, 6.0, 3)
    elif name == "ring":
        Z, X = wl.cyclocarbon_angstrom(6)
    elif name == "h2":
        Z, X = np.array([1, 1]), np.array([[0.0, 0, 0], [0, 0, 0.74]])
    else:  # one atom: the set is symmetric about every axis
        Z, X = np.array([1]), np.zeros((1, 3))
    return np.asarray(Z), np.asarray(X) * ca.ANGSTROM_TO_BOHR


@pytest.mark.parametrize("name", ["h", "h2", "h2o", "ring", "water9"])
def test_batches_and_weights(name):
    Z, X = _molecule(name)
    mol = ca.Molecule(Z, X, "cc-pvdz")
    P = ca.Grid(mol, "SG-1", 1, 0).points()
    assert np.array_equal(P, ca.Grid(mol, "SG-1", 1, 0).points())  # ties go by index: the same every time
    O = ol.OracleSystem(Z, X, "SG-1", "cc-pvdz").points()
    owner = np.full(len(P), len(Z))
    for a in reversed(np.flatnonzero(Z > 2)):
        owner[((P[:, :3] - X[a]) ** 2).sum(1) < CORE ** 2] = a
    assert np.all(np.diff(owner) >= 0)  # the atoms' core points first, then the rest
    for a in np.unique(owner):
        _check_split(P[owner == a, :3])
    # products of fewer than natoms factors (1 - m) / 2 whose m carries a few ulp each; a point is left out
    # when its weight is exactly 0, which the oracle's rounding may put at 1e-17 of the largest
    key = lambda A: [tuple(r) for r in np.round(A[:, :3] + 0.0, 7) + 0.0]
    w, top = dict(zip(key(O), O[:, 3])), O[:, 3].max()
    for k, v in zip(key(P), P[:, 3]):
        assert abs(w.pop(k) - v) <= 1e-12 * top
    assert all(abs(v) <= 1e-15 * top for v in w.values())
