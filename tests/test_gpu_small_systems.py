"""The splits of the work that depend on the number of atoms, at their edges.

  * Lennard-Jones: 8, 4, 2 or 1 lanes per atom up to 32,768, 65,536 and
    131,072 atoms and above, one and two species, against the oracle (FP64
    on both sides: 1e-10, as the other pair tests);
  * charge relaxation: one block finishes a step up to 8,192 atoms and runs
    ahead of the host from the third evaluation on; several kernels above.
    Zero to five steps, a stop by tolerance in each of them, and a run that
    diverges, against the same dynamics driven from outside.  The charges
    differ by the rounding of means and of the rates' few operations, so
    1e-12 of their range.
"""
import numpy as np
import pytest

from helpers import rel_maxnorm
from pysic_amd import structures as st
from pysic_amd.interactions import Potential, build_descriptors
from pysic_amd.learned import kcells

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    from pysic_amd.engine import Engine
    e = Engine(0)
    yield e
    e.close()


@pytest.mark.parametrize("n,species", [(1, 1), (37, 2), (32768, 1), (32769, 1), (32769, 2),
                                       (65536, 1), (65537, 2), (131072, 1), (131073, 1)])
def test_lennard_jones_lanes(eng, oracle, n, species):
    print("case: LJ lanes n=%d species=%d" % (n, species), flush=True)
    m = 4
    while 4 * m ** 3 < n:
        m += 1
    full = st.fcc((m, m, m), a=5.6, sigma=0.12, seed=n)
    keep = np.sort(np.random.default_rng(n).permutation(len(full))[:n])
    pos = full.positions[keep]
    sp = (np.arange(n) % species).astype(np.int32)
    names = ["Ar", "Kr"][:species]
    model = [Potential("LJ", symbols=[[a, b]], parameters=[0.2 + 0.1 * k, 3.1], cutoff=5.0,
                       cutoff_margin=0.5)
             for k, (a, b) in enumerate([("Ar", "Ar"), ("Kr", "Kr"), ("Ar", "Kr")][:2 * species - 1])]
    pd, bd, _ = build_descriptors(model, {x: k for k, x in enumerate(names)})
    cut = np.full(n, 5.2)
    eng.create_atoms(sp, pos)
    eng.create_cell(full.cell, (True, True, True))
    eng.set_potentials(pd)
    eng.set_bond_order_factors(np.zeros((0, 14)))
    eng.ewald_off()
    eng.generate_neighbor_lists(cut)
    nl = oracle.neighbor_list(pos, full.cell, [1, 1, 1], cut)
    args = (sp, pos, None, full.cell, nl, pd, np.zeros((0, 14)))
    e_ref = oracle.evaluate("energy", *args)
    f_ref, w_ref = oracle.evaluate("forces", *args)
    e = eng.energy()
    f, w = eng.forces()
    assert abs(e - e_ref) <= 1e-10 * max(1.0, abs(e_ref))
    assert np.abs(f - f_ref).max() <= 1e-10 * max(1.0, np.abs(f_ref).max())
    assert np.abs(w - w_ref).max() <= 1e-10 * max(1.0, np.abs(w_ref).max())


def _relaxation_case(eng, n):
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1.0 / 3.0) - 1e-9)) + (n < 8)
    g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    cell = np.diag([3.0 * m + 4.0] * 3)
    eng.create_atoms(np.zeros(n, np.int32), 3.0 * g + rng.normal(0.0, 0.05, (n, 3)),
                     charges=np.zeros(n))
    eng.create_cell(cell, (True, True, True))
    eng.set_potentials(np.array([[2, 1, 0, 0, 10.0, 2.0, 0, 0, -1, 0, 0, 0]]))
    eng.set_bond_order_factors(np.zeros((0, 14)))
    eng.set_ewald(4.0, 0.9, kcells(cell, 0.9), 1.5, 0.00552635)
    eng.generate_neighbor_lists(np.full(n, 4.2))
    return rng.normal(0.0, 0.1, n), rng.normal(0.0, 0.01, n)


def _driven(eng, q, v, n_steps, dt, fr, tol):
    def force():
        eng.update_charges(q)
        x = eng.electronegativities()
        return x - x.mean()
    f, steps, err = force(), 0, 2.0 * tol
    errs = []
    while err > tol and steps < n_steps:
        q = q + v * dt + (f - fr * v) * dt * dt
        v = (1 - 0.5 * fr * dt) * v + 0.5 * f * dt
        f = force()
        v = (v + 0.5 * f * dt) / (1 + 0.5 * fr * dt)
        steps, err = steps + 1, f.max()
        errs.append(err)
    return q, v, steps, err, errs


@pytest.mark.parametrize("n", [2, 1023, 1025, 8192, 8193])
def test_relaxation_steps_and_stops(eng, n):
    print("case: relaxation n=%d" % n, flush=True)
    q0, v0 = _relaxation_case(eng, n)
    dt, fr = 0.05, 4.0
    _, _, _, _, errs = _driven(eng, q0, v0, 5, dt, fr, 1e-300)
    assert all(a > b for a, b in zip(errs, errs[1:]))
    for n_steps, tol in [(0, 1e-9), (1, 1e-9), (2, 1e-9), (3, 1e-9), (5, 1e-9)] + [
            (5, 0.5 * (a + b)) for a, b in zip(errs, errs[1:])] + [(5, 2.0 * errs[0])]:
        q, v, steps, err, _ = _driven(eng, q0, v0, n_steps, dt, fr, tol)
        got, rate, k, e = eng.relax_charges(q0, v0, n_steps, dt, 1.0, fr, tol)
        assert k == steps
        assert abs(e - err) <= 1e-9 * abs(err)
        assert rel_maxnorm(got, q) <= 1e-12 and np.abs(rate - v).max() <= 1e-12


@pytest.mark.parametrize("tol", [0.0, -1e-9, float("nan"), float("inf")])
@pytest.mark.parametrize("n", [2, 8192, 8193])
def test_relaxation_that_is_not_entered(eng, n, tol):
    """The loop is entered while twice the tolerance is above the tolerance:
    with one that is zero, negative, infinite or not a number nothing moves."""
    print("case: relaxation n=%d tolerance %r" % (n, tol), flush=True)
    q0, v0 = _relaxation_case(eng, n)
    got, rate, k, e = eng.relax_charges(q0, v0, 5, 0.05, 1.0, 4.0, tol)
    assert k == 0
    assert np.array_equal(got, q0) and np.array_equal(rate, v0)
    assert np.array_equal(e, 2.0 * tol, equal_nan=True)
    # and the device's own copies are the caller's as well
    x = eng.electronegativities()
    eng.update_charges(q0)
    assert np.array_equal(eng.electronegativities(), x)


@pytest.mark.parametrize("n", [1023, 8193])
def test_relaxation_that_diverges_is_reported(eng, n):
    print("case: diverging relaxation n=%d" % n, flush=True)
    q0, v0 = _relaxation_case(eng, n)
    with pytest.raises(Exception, match="diverged"):
        eng.relax_charges(q0, v0, 5000, 5.0, 1.0, 0.0, 1e-9)
    # and the next relaxation starts clean
    got, _, k, _ = eng.relax_charges(q0, v0, 2, 0.05, 1.0, 4.0, 1e-9)
    q, _, _, _, _ = _driven(eng, q0, v0, 2, 0.05, 4.0, 1e-9)
    assert k == 2 and rel_maxnorm(got, q) <= 1e-12


@pytest.mark.parametrize("n", [864, 137388])
def test_image_words_follow_the_list_build(eng, n):
    """The Lennard-Jones kernels skip the image words of waves whose entries
    are all in the atom's own image, which only the lane-parallel build
    records: after any order of builds, and after dynamics, the forces are
    those of lists built atom by atom, bit for bit (up to 131,072 atoms the
    lanes sum in the list's order, which is the same)."""
    print("case: images n=%d" % n, flush=True)
    m = round((n / 4) ** (1.0 / 3.0))
    s = st.fcc((m, m, m), a=5.4, sigma=0.1, seed=6)
    assert len(s) == 4 * m ** 3
    n = len(s)
    pd, _, _ = build_descriptors([Potential("LJ", symbols=[["Ar", "Ar"]], parameters=[0.01, 3.4],
                                            cutoff=6.4)], {"Ar": 0})
    st.maxwell_boltzmann(s, 60.0, 2)
    eng.create_atoms(np.zeros(n, np.int32), s.positions, masses=s.masses, momenta=s.momenta)
    eng.create_cell(s.cell, (True, True, True))
    eng.set_potentials(pd)
    eng.set_bond_order_factors(np.zeros((0, 14)))
    eng.ewald_off()

    def forces(method):
        eng.set_neighbor_method(method)
        eng.generate_neighbor_lists(np.full(n, 6.6))
        return eng.forces()[0]
    want = forces(1)
    for method in (0, 1, 4, 0):
        assert np.array_equal(forces(method), want)
    for method in (0, 1, 0, 1):      # steps replayed from graphs, then lists of both kinds
        forces(method)
        eng.md_run(4, 0.5)
        f = eng.forces()[0]
        assert np.array_equal(forces(1), f) and np.array_equal(forces(0), f)
    eng.set_neighbor_method(0)
