"""The lane-parallel neighbor scan of one cell below 2^17 atoms and of any size
where bins are dense (its 27 bins as one stream) against the per-atom scan: the same lists entry by entry, in
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


@pytest.mark.parametrize("bins", [(16, 16, 32), (16, 17, 32), (32, 32, 16), (64, 32, 33)])
def test_lists_around_the_one_block_scan(oracle, bins):
    """The bins' scan is one block's work up to 8,192 of them."""
    from pysic_amd.engine import Engine
    n, rc = 6000, 2.5
    print("case: %d bins" % np.prod(bins), flush=True)
    cell = np.diag((np.array(bins) + 0.5) * rc)
    pos = np.random.default_rng(sum(bins)).random((n, 3)) @ cell
    eng = Engine(0)
    eng.create_atoms(np.zeros(n, np.int32), pos)
    eng.create_cell(cell)
    eng.set_potentials(np.zeros((0, 12)))
    eng.set_bond_order_factors(np.zeros((0, 14)))
    eng.ewald_off()
    for k in range(3):   # the third build follows two sorts with atoms changing bins
        p = pos + 1.3 * k
        eng.update_coordinates(p)
        eng.generate_neighbor_lists(np.full(n, rc))
        assert_same_pairs(eng, oracle.neighbor_list(p, cell, [1, 1, 1], np.full(n, rc)))
    eng.close()


def test_the_scan_of_many_bins_uses_the_chip():
    """A step of 140,608 atoms (64,000 bins) is no longer than one of 262,144
    (122,500 bins): in one block the scan alone took 40 of its 130 us."""
    import time
    from pysic_amd import structures as st
    from pysic_amd.engine import Engine
    from helpers import tersoff_descriptors
    pd, bd = tersoff_descriptors()
    step = {}
    for reps in ((26, 26, 26), (32, 32, 32)):
        s = st.maxwell_boltzmann(st.diamond_si(reps, sigma=0.1, seed=1), 600.0, 2)
        n = len(s)
        print("case: step of %d atoms" % n, flush=True)
        eng = Engine(0)
        eng.create_atoms(np.zeros(n, np.int32), s.positions, masses=s.masses, momenta=s.momenta)
        eng.create_cell(s.cell)
        eng.set_potentials(pd)
        eng.set_bond_order_factors(bd)
        eng.ewald_off()
        eng.generate_neighbor_lists(np.full(n, 3.5))
        times = []
        for _ in range(9):
            t = time.perf_counter()
            eng.md_run(40, 0.02, rebuild=1)
            times.append(time.perf_counter() - t)
        step[n] = np.median(times[2:]) / 40
        eng.close()
    print({n: round(1e6 * t, 1) for n, t in step.items()}, flush=True)
    assert step[140608] < step[262144]


@pytest.mark.parametrize("pbc", [(1, 1, 1), (0, 0, 0)])
def test_dense_bins_are_not_one_threads_work(pbc):
    """Where bins are dense, the per-atom prefiltered scan asked for by its
    number is the lane-parallel one: the default's lists, entry by entry, in
    the default's time (a thread per atom takes 10 to 20 times as long)."""
    from pysic_amd import structures as st
    from pysic_amd.engine import Engine
    s = st.fcc((16, 16, 16), a=5.26, sigma=0.05, seed=1)
    n = len(s)
    times, lists = {}, {}
    for method in (0, 5):
        print("case: method %d pbc %s" % (method, pbc), flush=True)
        eng = Engine(0)
        eng.create_atoms(np.zeros(n, np.int32), s.positions)
        eng.create_cell(s.cell, pbc)
        eng.set_potentials(np.zeros((0, 12)))
        eng.set_bond_order_factors(np.zeros((0, 14)))
        eng.ewald_off()
        eng.set_neighbor_method(method)
        eng.generate_neighbor_lists(np.full(n, 9.0))
        lists[method] = eng.neighbor_lists()
        eng.timing(True)
        for _ in range(10):
            eng.generate_neighbor_lists(np.full(n, 9.0))
        ms, calls = eng.timing_read()["neighbors"]
        times[method] = ms / calls
        eng.close()
    for x, y in zip(lists[0], lists[5]):
        assert np.array_equal(x, y)
    print(times, flush=True)
    assert times[5] < 3.0 * times[0]
