"""The lane-parallel neighbor scan of one cell below 2^17 atoms (and any size where bins are dense; its 27 bins
as one stream) against the per-atom scan: the same lists entry by entry, in
the same order, and the oracle's as sets.  Cells of one, two and more bins an
axis, open axes with atoms outside the box, atoms several cells away, sparse
and dense bins (8 and 16 lanes an atom), and per-atom radii."""
import numpy as np
import pytest

from helpers import assert_same_pairs

pytestmark = pytest.mark.gpu

CASES = [
    # (atoms, edges over the radius, pbc, radius spread, cells away)
    (1, (3.0, 3.0, 3.0), (1, 1, 1), 0.0, 0),
    (7, (1.0, 1.5, 1.0), (1, 1, 1), 0.0, 0),        # one bin an axis: own images
    (63, (2.2, 1.1, 3.4), (1, 1, 1), 0.0, 2),
    (257, (4.0, 5.0, 6.0), (1, 1, 1), 0.3, 1),       # sparse, per-atom radii
    (500, (4.5, 5.5, 3.5), (0, 1, 0), 0.0, 0),      # open axes, atoms outside
    (401, (6.0, 4.0, 5.0), (0, 0, 0), 0.2, 0),
    (1500, (3.3, 3.9, 4.2), (1, 1, 1), 0.0, 3),      # dense bins: 16 lanes
    (900, (2.0, 2.9, 2.1), (1, 0, 1), 0.1, 0),
    (4096, (9.0, 8.0, 7.0), (1, 1, 1), 0.0, 0),
]


@pytest.mark.parametrize("k", range(len(CASES)))
def test_lists_are_the_per_atom_scans(oracle, k):
    from pysic_amd.engine import Engine
    n, edges, pbc, spread, away = CASES[k]
    rng = np.random.default_rng(50 + k)
    rc = 2.5
    cell = np.diag(np.array(edges) * rc) + rng.uniform(-0.1, 0.1, (3, 3)) * (k % 2)
    # bins are cut along the perpendicular widths: keep them above the radius
    for a in range(3):
        if np.abs(np.linalg.det(cell)) / np.linalg.norm(
                np.cross(cell[(a + 1) % 3], cell[(a + 2) % 3])) < rc:
            cell[a] *= 1.3
    u = rng.random((n, 3))
    for a in range(3):
        if pbc[a]:
            u[:, a] += rng.integers(-away, away + 1, n)
        else:
            u[:, a] = u[:, a] * 1.3 - 0.15
    pos = u @ cell
    cut = rc * (1.0 - spread * rng.random(n))
    cut[0] = rc
    got = {}
    for method in (0, 1):
        eng = Engine(0)
        eng.create_atoms(np.zeros(n, np.int32), pos)
        eng.create_cell(cell, pbc)
        eng.set_potentials(np.zeros((0, 12)))
        eng.set_bond_order_factors(np.zeros((0, 14)))
        eng.ewald_off()
        eng.set_neighbor_method(method)
        eng.generate_neighbor_lists(cut)
        got[method] = eng.neighbor_lists()
        if method == 0:
            nl = oracle.neighbor_list(pos, cell, list(pbc), cut)
            assert_same_pairs(eng, nl)
        eng.close()
    for x, y in zip(got[0], got[1]):
        assert np.array_equal(x, y)
